"""Thin and flat boxes, whose tiles two steps per launch would leave mostly empty, keep single
steps (one array for an AA box, as its device memory shows), boxes next to them take pairs,
and both give the states of single steps."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice

pytestmark = pytest.mark.gpu

CASES = [  # size, storage, D3Q, pairs
    ((512, 1, 512), "f64", 19, False), ((128, 2, 256), "f64", 27, False), ((128, 3, 256), "f64", 19, True),
    ((512, 9, 64), "f32s", 19, False), ((512, 9, 64), "f64", 19, True), ((512, 11, 64), "f32s", 27, True),
    ((128, 3, 256), "f32s", 19, False), ((128, 4, 256), "f32s", 19, True),
    ((512, 512, 2), "f64", 19, False), ((512, 512, 3), "f64", 19, True), ((512, 512, 3), "f64", 27, False),
    ((512, 512, 3), "f32s", 19, False), ((512, 512, 4), "f32s", 19, True), ((256, 256, 1), "f64", 19, True),
    ((100000, 1, 1), "f32s", 27, False), ((128, 128, 16), "f16s", 19, False), ((320, 100, 90), "f16s", 27, False),
    ((120, 17, 300), "f16s", 19, False), ((80, 80, 80), "f16s", 27, True),
    ((64, 64, 12), "f32s", 19, False), ((79, 14, 47), "f64", 19, False), ((32, 32, 32), "f32s", 27, True),
]


@pytest.mark.parametrize("size, storage, q, pairs", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_thin_boxes(size, storage, q, pairs, monkeypatch):
    print(f"[thin] {size} {storage} {q}", flush=True)
    one = q * {"f64": 8, "f32s": 4, "f16s": 2}[storage] * size[0] * size[1] * size[2]
    out = []
    for env in (None, "0"):
        if env:
            monkeypatch.setenv("LBM_DENSE_PAIR", env)
        with DenseLattice(*size, q=q, storage=storage, omega=1 / 0.8) as lat:
            if env is None:
                assert (lat.info()["device_bytes"] > 2 * one) == pairs
            lat.init_tgv(0.03, 1e-3, 3)
            lat.step(3)
            out.append(lat.moments())
    assert all(np.array_equal(a, b) for a, b in zip(*out))
