"""Large readbacks (staged through pinned memory) equal the state that small ones
give: sizes that end inside a chunk, a piece and a 16-byte word, repeated, and
after a small first copy; FP32 adjoint states converted on the way."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import Adjoint, DenseLattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(128, 100, 113), (161, 97, 61), (64, 64, 64), (129, 111, 127)],
                         ids=lambda s: "x".join(map(str, s)))
def test_large_readback_equals_parts(size):
    nx, ny, nz = size
    print(f"[readback] {size}", flush=True)
    rng = np.random.default_rng(3)
    n = nx * ny * nz
    f = 0.05 + 0.01 * rng.random((19, n))
    with DenseLattice(nx, ny, nz) as lat:
        for _ in range(2):
            lat.set_state(f)
            assert np.array_equal(lat.get_state(), f)  # 19 n doubles
            rho, u = lat.moments()
            want = f[0].copy()  # the sum in slot order, as the readout forms it
            for s in range(1, 19):
                want += f[s]
            assert np.array_equal(rho, want)
            assert np.allclose(u[:, 0] * rho, f[[0, 6, 7, 8, 9]].sum(0) - f[[1, 10, 11, 12, 13]].sum(0),
                               rtol=0, atol=1e-15)


def test_large_adjoint_states_f32():
    """An FP32 adjoint state above the size that is staged from the first copy on (32 MiB of
    floats), not a multiple of a chunk, piece or word, against the FP64 adjoint cell by cell: the
    state is random, so a piece put in another place differs by as much as the values."""
    size = (101, 97, 53)
    n = size[0] * size[1] * size[2]
    assert 19 * n * 4 > 32 << 20 and 19 * n * 4 % (1 << 20) and 19 * n * 4 % 16
    f = 0.05 + 0.01 * np.random.default_rng(5).random((19, n))
    lam = {}
    for storage in ("f64", "f32s"):
        with Adjoint(*size, storage=storage, gamma=np.zeros(n), checkpoint_every=2) as adj:
            adj.set_initial_state(f)
            print(f"[readback] adjoint {storage}", flush=True)
            adj.forward(2)
            adj.backward()
            lam[storage] = adj.lambda0()
            assert np.array_equal(adj.lambda0(), lam[storage])
    big = np.abs(lam["f64"]).max()
    assert np.array_equal(lam["f32s"], lam["f32s"].astype(np.float32))
    # two steps of some tens of FP32 operations: a few tens of ulps of the largest value
    assert np.abs(lam["f32s"] - lam["f64"]).max() <= 64 * 2.0 ** -24 * big
    assert np.abs(np.diff(lam["f64"].reshape(-1))).mean() > 1e-2 * big
