"""Two steps per launch with stores that stream past the caches (LBM_DENSE_NT=1, what large boxes
take) at the sizes where tiles, chunks and walls meet: masked boxes and split rows against single
cached steps, bit for bit."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 3, 1), (32, 16, 5), (33, 17, 2), (63, 8, 4), (65, 7, 6), (130, 20, 11), (24, 37, 40)]


def states(monkeypatch, size, **kw):
    out = []
    for pair, nt in ("11", "00"):
        monkeypatch.setenv("LBM_DENSE_PAIR", pair)
        monkeypatch.setenv("LBM_DENSE_NT", nt)
        with DenseLattice(*size, omega=1 / 0.6, **kw) as lat:
            lat.init_tgv(0.05, 1e-3, 3)
            lat.step(5)
            out.append((lat.get_state(), *lat.moments(), lat.mass()))
    return out


def same(out):
    assert all(np.array_equal(a, b) for a, b in zip(out[0][:3], out[1][:3]))
    assert abs(out[0][3] - out[1][3]) <= 1e-12 * abs(out[1][3])


@pytest.mark.parametrize("periodic", [(1, 1, 1), (1, 0, 1), (0, 0, 0), (0, 1, 1)],
                         ids=lambda p: "".join(map(str, p)))
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_masked_pairs_streaming(size, periodic, monkeypatch):
    ncell = size[0] * size[1] * size[2]
    solid = (O.uniform01(7, np.arange(ncell, dtype=np.uint64)) < 0.3).astype(np.uint8)
    for mask in (None, solid):
        if (mask is None and periodic == (1, 1, 1)) or (mask is not None and mask.all()):
            continue
        for q, storage, force in ((19, "f64", 0.0), (19, "f64", 1e-4), (19, "f32s", 1e-4), (27, "f32s", 0.0)):
            print(f"[streaming] masked {size} {periodic} {mask is not None} {q} {storage}", flush=True)
            same(states(monkeypatch, size, q=q, storage=storage, solid=mask, periodic=periodic, pattern="ab",
                        pull=True, force=(force, 0.0, -force),
                        density_jump_x=3e-3 if periodic[0] else 0.0))


@pytest.mark.parametrize("size", [(2, 3, 1), (4, 16, 5), (64, 9, 3), (66, 17, 2), (128, 8, 4), (130, 7, 6),
                                  (260, 20, 9), (48, 37, 40)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("q, storage", [(19, "f16s"), (27, "f16s"), (19, "f32s")])
def test_split_rows_streaming(q, storage, size, monkeypatch):
    monkeypatch.setenv("LBM_DENSE_PAIR_CELLS", "2")
    for force in (0.0, 1e-4):
        print(f"[streaming] split {size} {q} {storage} {force}", flush=True)
        same(states(monkeypatch, size, q=q, storage=storage, force=(force, -force, 0.0)))
