"""FP32 and FP16 deviation steps, rounding by rounding: single steps and two steps per
launch against the collision restated in numpy with every float operation and FMA in its
place.  (An FMA is taken in 64-bit-mantissa arithmetic and rounded to FP32: the product is
exact, and the sum's first rounding decides the second with a chance of about 2^-39.)"""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice
from oracle import oracle as O

pytestmark = pytest.mark.gpu

f32 = np.float32


def fma(a, b, c):
    wide = np.longdouble
    return (np.asarray(a, wide) * np.asarray(b, wide) + np.asarray(c, wide)).astype(f32)


def collide(d, c, w, omega, force, f16):
    """d[Q, n] FP32 deviations before the collision -> after it."""
    q = len(d)
    drho, m = np.zeros(d.shape[1]), np.zeros((3, d.shape[1]))
    for s in range(q):
        x = d[s].astype(np.float64)
        drho = drho + x
        for k in range(3):
            if c[s][k]:
                m[k] = m[k] + c[s][k] * x
    rho = 1.0 + drho
    forced = any(force)
    u = [((m[k] + 0.5 * force[k]) if forced else m[k]) * (1.0 / rho) for k in range(3)]
    u = [x.astype(f32) for x in u]
    F = [f32(x) for x in force]
    uu = f32(3) * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    fu = f32(3) * (F[0] * u[0] + F[1] * u[1] + F[2] * u[2])
    om = f32(omega)
    omf, keep = f32(1) - f32(0.5) * om, f32(1) - om
    drho, rho = drho.astype(f32), rho.astype(f32)

    def along(v, s):  # c_s . v, terms in order
        total = None
        for k in range(3):
            if c[s][k]:
                t = v[k] if c[s][k] > 0 else -v[k]
                total = t if total is None else total + t
        return total

    out = np.empty_like(d)
    for s in range(q):
        if any(c[s]):
            cu = f32(3) * along(u, s)
            e = fma(f32(0.5) * cu, cu, cu) - f32(0.5) * uu
            sf = along(F, s)
            fd = fma(cu, f32(3) * sf, fma(f32(3), sf, -fu))
        else:
            e, fd = -(f32(0.5) * uu), -fu
        eqdev = fma(rho, e, drho)
        if not forced:
            x = om * eqdev
        elif f16:
            x = fma(omf, fd, om * eqdev)
        else:
            x = fma(om, eqdev, omf * fd)
        out[s] = fma(keep, d[s], f32(w[s]) * x)
    return out


@pytest.mark.parametrize("force", [(0.0, 0.0, 0.0), (1e-4, -2e-4, 3e-4)], ids=["f0", "force"])
@pytest.mark.parametrize("storage", ["f32s", "f16s"])
@pytest.mark.parametrize("q", [19, 27])
def test_deviation_steps_round_as_written(q, storage, force, monkeypatch):
    nx, ny, nz = 34, 9, 6
    n, steps, omega, scale = nx * ny * nz, 4, 1 / 0.6, f32(4096)
    c, _, w = O.lattice(q)
    rng = np.random.default_rng(q)
    d = rng.uniform(-1e-3, 1e-3, (q, n)).astype(f32)
    if storage == "f16s":
        d = (d * scale).astype(np.float16).astype(f32) / scale
    start = d.astype(np.float64) + w[:, None]
    for _ in range(steps):
        d = collide(d, c, w, omega, force, storage == "f16s")
        if storage == "f16s":
            d = (d * scale).astype(np.float16).astype(f32) / scale
        for s in range(q):
            d[s] = np.roll(d[s].reshape(nz, ny, nx), (c[s][2], c[s][1], c[s][0]), (0, 1, 2)).ravel()
    for pair in "01":
        for pattern, pull in (("aa", False), ("ab", True), ("ab", False)):
            print(f"[rounding] q={q} {storage} {force} pair={pair} {pattern} {pull}", flush=True)
            monkeypatch.setenv("LBM_DENSE_PAIR", pair)
            with DenseLattice(nx, ny, nz, q=q, pattern=pattern, pull=pull, storage=storage,
                              omega=omega, force=force) as lat:
                lat.set_state(start)
                lat.step(steps)
                got = (lat.get_state() - w[:, None]).astype(f32)
            assert np.array_equal(got, d)
