"""The drop-in kernels on the compressed adjacency (LBM_SPARSE_COMPRESS=1) equal
the oracle bit for bit: lists whose groups of 64 compress (box, channel), lists
with groups that do not (random solids, short rows), lengths around multiples of
64, and launches over ranges that start and end inside a group."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_dense import seeded_fc
from tests.test_gpu_sparse import run_gpu

pytestmark = pytest.mark.gpu


def geometry(name):
    if name == "box":
        return O.DenseGeometry(20, 9, 13, order="reference")
    if name == "single":
        return O.DenseGeometry(1, 1, 63)
    if name == "group":
        return O.DenseGeometry(8, 8, 1)
    if name == "channel":
        nx, ny, nz = 11, 17, 70
        solid = np.zeros((nz, ny, nx), np.uint8)
        solid[:, 0] = solid[:, -1] = 1
        solid[20:25, 5:9, 3:6] = 1
        return O.DenseGeometry(nx, ny, nz, solid.reshape(-1), periodic=(1, 0, 1), order="reference")
    nx, ny, nz = 16, 15, 14
    solid = (O.uniform01(9, np.arange(nx * ny * nz, dtype=np.uint64)) < 0.3).astype(np.uint8)
    return O.DenseGeometry(nx, ny, nz, solid, periodic=(0, 1, 1), order="reference")


@pytest.mark.parametrize("name", ["box", "single", "group", "channel", "random"])
@pytest.mark.parametrize("layout", ["soa", "aos"])
@pytest.mark.parametrize("q", [19, 27])
def test_compressed_adjacency_equals_oracle(q, layout, name, monkeypatch):
    monkeypatch.setenv("LBM_SPARSE_COMPRESS", "1")
    g = geometry(name)
    n, L = g.nfluid, O.SOA if layout == "soa" else O.AOS
    fc = seeded_fc(g, q)
    omega, splits = 1 / 0.6, sorted({min(n, 5), n // 3, n // 2 + 1})
    for prec, dt in (("f64", np.float64), ("f32", np.float32)):
        print(f"[compressed] q={q} {layout} {name} {prec} n={n}", flush=True)
        adj = g.adjacency(q, L, O.ADJ_PULL)
        f0 = O.to_storage(fc, q, L, aa_even_ready=True).astype(dt)
        want = f0.copy()
        O.run_aa(q, L, n, want, adj, 5, omega)
        assert np.array_equal(run_gpu(q, layout, prec, omega, adj, f0, 5, "aa", splits=splits), want)
        f0 = O.to_storage(fc, q, L).astype(dt)
        if layout == "soa":
            want = O.run_ab(q, L, n, f0, adj, 3, omega, pull=True)
            assert np.array_equal(run_gpu(q, layout, prec, omega, adj, f0, 3, "ab", pull=True,
                                          splits=splits), want)
        adj = g.adjacency(q, L, O.ADJ_PUSH)
        want = O.run_ab(q, L, n, f0, adj, 3, omega)
        assert np.array_equal(run_gpu(q, layout, prec, omega, adj, f0, 3, "ab", adjacency_mode=0,
                                      splits=splits), want)
