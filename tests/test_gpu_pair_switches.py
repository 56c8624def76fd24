"""Switches that meet: two steps per launch asked for together with interleaved rows
(LBM_DENSE_PAIR=1 and LBM_DENSE_IROWS=1) give the states of single steps; a variable that
tunes the single-step kernels gives single steps."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice
from oracle import oracle as O
from tests.test_gpu_dense import seeded_fc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32s", "f16s"])
@pytest.mark.parametrize("masked", [False, True])
def test_pairs_with_interleaved_rows_asked_for(storage, masked, monkeypatch):
    size = (128, 11, 7)
    n = size[0] * size[1] * size[2]
    solid = (O.uniform01(7, np.arange(n, dtype=np.uint64)) < 0.3).astype(np.uint8) if masked else None
    g = O.DenseGeometry(*size, solid)
    f = np.zeros((19, n))
    f[:, g.cell_of_fluid] = seeded_fc(g, 19)
    out = []
    for pair, irows in (("1", "1"), ("0", "0")):
        monkeypatch.setenv("LBM_DENSE_PAIR", pair)
        monkeypatch.setenv("LBM_DENSE_IROWS", irows)
        monkeypatch.setenv("LBM_DENSE_PAIR_CELLS", "2")
        print(f"[switches] {storage} masked={masked} pair={pair} irows={irows}", flush=True)
        with DenseLattice(*size, storage=storage, solid=solid, omega=1 / 0.8) as lat:
            lat.set_state(f)
            lat.step(5)
            out.append((lat.get_state(), *lat.moments(), lat.mass()))
    assert all(np.array_equal(a, b) for a, b in zip(out[0][:3], out[1][:3]))
    assert abs(out[0][3] - out[1][3]) <= 1e-12 * out[1][3]


@pytest.mark.parametrize("name, value", [
    ("BLOCK_X", "128"), ("BLOCKS_PER_CU", "4"), ("EVEN_BLOCK_X", "64"), ("EVEN_BLOCKS_PER_CU", "4"),
    ("ODD_IR_BLOCK_X", "64"), ("ODD_IR_BLOCKS_PER_CU", "4"), ("ODD_SEG_BLOCKS_PER_CU", "4"), ("STAGED", "2")])
def test_tuning_single_steps_asks_for_them(name, value, monkeypatch):
    """An AA box of one array, as its device memory shows."""
    one = 19 * 8 * 64 ** 3
    with DenseLattice(64, 64, 64) as lat:
        assert lat.info()["device_bytes"] > 2 * one
    monkeypatch.setenv("LBM_DENSE_" + name, value)
    with DenseLattice(64, 64, 64) as lat:
        assert lat.info()["device_bytes"] < 2 * one


@pytest.mark.parametrize("scale, pairs", [(1000.0, False), (4096.0, True), (1024.0, True)])
def test_fp16_pairs_need_a_power_of_two(scale, pairs, monkeypatch):
    """The two-step kernel works on scaled values; another scale takes single steps (one array)."""
    size, out = (66, 10, 9), []
    one = 19 * 2 * size[0] * size[1] * size[2]
    for pair in "10":
        monkeypatch.setenv("LBM_DENSE_PAIR", pair)
        print(f"[switches] f16 scale {scale} pair={pair}", flush=True)
        with DenseLattice(*size, storage="f16s", f16_scale=scale, omega=1 / 0.8) as lat:
            assert (lat.info()["device_bytes"] > 2 * one) == (pairs and pair == "1")
            lat.init_tgv(0.05, 1e-3, 3)
            lat.step(5)
            out.append((lat.get_state(), *lat.moments()))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
