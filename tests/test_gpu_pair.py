"""Two time steps per launch (LBM_DENSE_PAIR=1) against the oracle, and against
one step per launch (LBM_DENSE_PAIR=0), bit for bit: sizes at the edges of the
tiles (64 x 8, 64 x 4, 32 x 16, 32 x 8 cells, chunks along z), rows and columns
that wrap onto themselves, odd step counts, and graphs."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice
from oracle import oracle as O
from tests.test_gpu_dense import oracle_run, seeded_fc
from tests.test_gpu_graph import _Stream

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 3, 1), (32, 16, 5), (33, 17, 2), (31, 15, 3), (63, 8, 4), (64, 9, 3),
         (65, 7, 6), (130, 20, 11), (24, 37, 40)]


def run(monkeypatch, pair, size, fc, steps, **kw):
    monkeypatch.setenv("LBM_DENSE_PAIR", pair)
    with DenseLattice(*size, **kw) as lat:
        lat.set_state(fc)
        lat.step(steps)
        return lat.get_state()


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("q", [19, 27])
def test_pairs_equal_oracle_f64(q, size, monkeypatch):
    g = O.DenseGeometry(*size)
    fc = seeded_fc(g, q)
    for pattern, force, nt in (("aa", (0.0, 0.0, 0.0), "0"), ("push", (1e-4, -2e-4, 3e-4), "1"),
                               ("pull", (0.0, 0.0, 1e-4), "1")):
        monkeypatch.setenv("LBM_DENSE_NT", nt)
        print(f"[pair] q={q} {size} {pattern}", flush=True)
        got = run(monkeypatch, "1", size, fc, 5, q=q, pattern="aa" if pattern == "aa" else "ab",
                  pull=pattern == "pull", omega=1 / 0.6, force=force)
        assert np.array_equal(got, oracle_run(g, q, fc, pattern, 5, 1 / 0.6, force))


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("q", [19, 27])
def test_pairs_equal_single_steps_f32(q, size, monkeypatch):
    fc = seeded_fc(O.DenseGeometry(*size), q)
    for force in ((0.0, 0.0, 0.0), (1e-4, -2e-4, 3e-4)):
        print(f"[pair] f32s q={q} {size} {force}", flush=True)
        a, b = (run(monkeypatch, p, size, fc, 5, q=q, storage="f32s", omega=1 / 0.6, force=force)
                for p in "01")
        assert np.array_equal(a, b)


@pytest.mark.parametrize("size", [(2, 3, 1), (4, 16, 5), (64, 9, 3), (66, 17, 2), (128, 8, 4),
                                  (130, 7, 6), (260, 20, 9), (48, 37, 40)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("q, storage", [(19, "f16s"), (27, "f16s"), (19, "f32s")])
def test_split_rows_equal_single_steps(q, storage, size, monkeypatch):
    """Two cells per lane (split rows): states, moments and mass, through an odd step count and
    back in through set_state."""
    fc = seeded_fc(O.DenseGeometry(*size), q)
    monkeypatch.setenv("LBM_DENSE_PAIR_CELLS", "2")
    for force in ((0.0, 0.0, 0.0), (1e-4, -2e-4, 3e-4)):
        print(f"[pair] split {storage} q={q} {size} {force}", flush=True)
        out = []
        for pair in "01":
            monkeypatch.setenv("LBM_DENSE_PAIR", pair)
            with DenseLattice(*size, q=q, pattern="ab", pull=True, storage=storage, omega=1 / 0.6,
                              force=force) as lat:
                lat.set_state(fc)
                lat.step(5)
                lat.set_state(lat.get_state())
                lat.step(4)
                out.append((lat.get_state(), *lat.moments(), lat.mass()))
        assert all(np.array_equal(a, b) for a, b in zip(out[0][:3], out[1][:3]))
        assert abs(out[0][3] - out[1][3]) <= 1e-12 * out[0][3]


@pytest.mark.parametrize("periodic", [(1, 1, 1), (1, 0, 1), (0, 0, 0), (0, 1, 1), (1, 1, 0)],
                         ids=lambda p: "".join(map(str, p)))
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_masked_pairs(size, periodic, monkeypatch):
    """Walls and random solids, against the oracle (FP64) and single steps (FP32, pressure drop);
    the state, the mass and the moments read back through walls."""
    ncell = size[0] * size[1] * size[2]
    solid = (O.uniform01(7, np.arange(ncell, dtype=np.uint64)) < 0.3).astype(np.uint8)
    for mask in (None, solid):
        if mask is None and periodic == (1, 1, 1):
            continue
        if mask is not None and mask.all():
            continue
        g = O.DenseGeometry(*size, mask, periodic=periodic)
        fc = seeded_fc(g, 19)
        full = np.zeros((19, ncell))
        full[:, g.cell_of_fluid] = fc
        for pattern, force in (("pull", (0.0, 0.0, 0.0)), ("aa", (1e-4, -2e-4, 3e-4))):
            print(f"[pair] masked {size} {periodic} {mask is not None} {pattern}", flush=True)
            got = run(monkeypatch, "1", size, full, 5, pattern="aa" if pattern == "aa" else "ab",
                      pull=pattern == "pull", omega=1 / 0.6, force=force, solid=mask, periodic=periodic)
            want = np.zeros_like(full)
            want[:, g.cell_of_fluid] = oracle_run(g, 19, fc, pattern, 5, 1 / 0.6, force)
            assert np.array_equal(got, want)
        for q in (19, 27):
            out = []
            for pair in "01":
                monkeypatch.setenv("LBM_DENSE_PAIR", pair)
                with DenseLattice(*size, q=q, pattern="ab", pull=True, storage="f32s", omega=1 / 0.6,
                                  solid=mask, periodic=periodic,
                                  density_jump_x=3e-3 if periodic[0] else 0.0) as lat:
                    lat.init_tgv(0.05, 1e-3, 3)
                    lat.step(5)
                    out.append((lat.get_state(), *lat.moments(), lat.mass()))
            assert all(np.array_equal(a, b) for a, b in zip(out[0][:3], out[1][:3]))
            assert abs(out[0][3] - out[1][3]) <= 1e-12 * out[0][3]


def test_pairs_grouping_and_graphs(monkeypatch):
    """However the steps are grouped, and replayed from either array, the states are the same."""
    size, q = (70, 20, 9), 19
    fc = seeded_fc(O.DenseGeometry(*size), q)
    monkeypatch.setenv("LBM_DENSE_PAIR", "1")
    stream = _Stream()
    try:
        with DenseLattice(*size, omega=1 / 0.6) as a, DenseLattice(*size, omega=1 / 0.6) as b, \
                DenseLattice(*size, omega=1 / 0.6) as c:
            c.set_stream(stream.s.value)
            for lat in (a, b, c):
                lat.set_state(fc)
            with b.graph(6) as g:
                for n in (1, 3, 2):
                    for _ in range(n):
                        a.step(1)
                    b.step(n)
                    assert np.array_equal(a.get_state(), b.get_state())
                for _ in range(3):  # six steps from capture: odd numbers of pairs before and in it
                    g.launch()
                    a.step(3)
                    a.step(3)
                    assert np.array_equal(a.get_state(), b.get_state())
                    b.step(2)
                    a.step(1)
                    a.step(1)
            # a caller's own graph of an even run: every replay goes on where the last one ended
            graph, exe = stream.capture(lambda: c.step(2))
            for _ in range(5):
                stream.launch(exe)
            stream.synchronize()
            monkeypatch.setenv("LBM_DENSE_PAIR", "0")
            with DenseLattice(*size, omega=1 / 0.6) as d:
                d.set_state(fc)
                d.step(10)
                assert np.array_equal(c.get_state(), d.get_state())
            stream.destroy_graph(graph, exe)
    finally:
        stream.close()
