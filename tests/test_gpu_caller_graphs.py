"""A caller's own graph of an even run, replayed with other calls between the replays (eager
runs of even and odd length, single steps, a graph of the library's, new states), on handles
that take two steps per launch: the states equal those of a handle that takes single steps."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice
from oracle import oracle as O
from tests.test_gpu_dense import seeded_fc
from tests.test_gpu_graph import _Stream

pytestmark = pytest.mark.gpu

SIZE = (70, 20, 9)
BOXES = {
    "f64": dict(pattern="aa"),
    "split_f32": dict(pattern="ab", pull=True, storage="f32s"),
    "split_f16": dict(pattern="aa", storage="f16s"),
    "masked": dict(pattern="aa", masked=True, periodic=(1, 0, 1), force=(1e-5, 0.0, 0.0)),
    "masked_pull_f32": dict(pattern="ab", pull=True, storage="f32s", masked=True),
}


@pytest.mark.parametrize("warm", [0, 2, 3, 1])
@pytest.mark.parametrize("captured", [2, 4, 6])
@pytest.mark.parametrize("name", BOXES)
def test_replays_between_other_calls(name, captured, warm, monkeypatch):
    kw = dict(BOXES[name])
    ncell = SIZE[0] * SIZE[1] * SIZE[2]
    if kw.pop("masked", False):
        kw["solid"] = (O.uniform01(7, np.arange(ncell, dtype=np.uint64)) < 0.2).astype(np.uint8)
    if name.startswith("split"):
        monkeypatch.setenv("LBM_DENSE_PAIR_CELLS", "2")
    f = 0.05 + 0.001 * np.random.default_rng(3).random((19, ncell))
    if "solid" in kw:
        f[:, kw["solid"] != 0] = 0.0
    lats = []
    for pair in "10":
        monkeypatch.setenv("LBM_DENSE_PAIR", pair)
        lats.append(DenseLattice(*SIZE, omega=1 / 0.8, **kw))
    a, b = lats
    stream = _Stream()
    try:
        print(f"[caller graph] {name} captured={captured} warm={warm}", flush=True)
        a.set_stream(stream.s.value)
        for lat in lats:
            lat.set_state(f)
            lat.step(warm)
        graph, exe = stream.capture(lambda: a.step(captured))
        own = a.graph(6)

        def replay():
            stream.launch(exe)
            b.step(captured)

        def both(call):
            call(a)
            call(b)

        def own_graph():
            own.launch()
            b.step(6)

        def same(where):
            assert np.array_equal(a.get_state(), b.get_state()), where
            assert all(np.array_equal(x, y) for x, y in zip(a.moments(), b.moments())), where

        same("capture runs nothing")
        for where, call in (
                ("eager 2", lambda: both(lambda lat: lat.step(2))),
                ("eager 3, 1", lambda: both(lambda lat: (lat.step(3), lat.step(1)))),
                ("eager 6", lambda: both(lambda lat: lat.step(6))),
                ("eager 1, 1", lambda: both(lambda lat: (lat.step(1), lat.step(1)))),
                ("own graph", own_graph), ("own graph again", own_graph),
                ("timed", lambda: both(lambda lat: lat.run_timed(2))),
                ("nothing", lambda: None)):
            replay()
            same("replay before " + where)
            call()
            same(where)
            replay()
            replay()
            same("replay after " + where)
        if warm % 2 == 0:  # (a new state is at step 0, which a graph of odd phase does not continue)
            for where, call in (("set_state", lambda lat: lat.set_state(f)),
                                ("init", lambda lat: lat.init_tgv(0.03, 1e-4, 5))):
                both(lambda lat: lat.step(2))
                both(call)
                replay()
                same(where)
                both(lambda lat: lat.step(1))
                both(call)
                replay()
                both(lambda lat: lat.step(2))
                replay()
                same(where + " after an odd step")
        own.close()
        stream.synchronize()
        stream.destroy_graph(graph, exe)
    finally:
        for lat in lats:
            lat.close()
        stream.close()
