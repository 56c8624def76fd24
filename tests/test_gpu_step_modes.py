"""Handles that take two steps per launch go back to their own way of stepping for calls of one
step in a row, and into pairs again for longer calls: whatever the calls, the states are those
of a handle that never takes pairs, and a state set is the state read back."""
import numpy as np
import pytest

from lbmminiapp_amd.capi import DenseLattice
from oracle import oracle as O
from tests.test_gpu_graph import _Stream

pytestmark = pytest.mark.gpu

SMALL = (70, 20, 11)
BOXES = {
    "pull_walls_f64": (SMALL, dict(pattern="ab", pull=True, masked=True, force=(1e-5, 0.0, 0.0))),
    "pull_walls_jump_f32": (SMALL, dict(pattern="ab", pull=True, masked=True, storage="f32s", jump=3e-3)),
    "push_jump_f64": (SMALL, dict(pattern="ab", masked=True, jump=3e-3)),
    "push_f32": (SMALL, dict(pattern="ab", masked=True, storage="f32s", periodic=(1, 0, 0))),
    "aa_walls_f64": (SMALL, dict(masked=True, periodic=(0, 0, 1))),
    "aa_jump_f64": (SMALL, dict(masked=True, jump=3e-3)),
    "aa_jump_f32_q27": (SMALL, dict(masked=True, jump=3e-3, storage="f32s", q=27)),
    "push_gather_jump_f64": (SMALL, dict(pattern="ab", masked=True, jump=3e-3, gather=True)),
    "pull_split_f16": (SMALL, dict(pattern="ab", pull=True, storage="f16s")),
    "push_split_f32": (SMALL, dict(pattern="ab", storage="f32s")),
    # AA in place where two arrays exceed the memory-side cache: interleaved rows, plain ones
    "aa_f64_128": ((128, 128, 80), dict()),
    "aa_f16_rows": ((256, 192, 150), dict(storage="f16s")),
    "aa_f32_q27_odd": ((101, 113, 120), dict(storage="f32s", q=27, force=(0.0, 1e-5, 0.0))),
    "aa_walls_jump_f64": ((128, 100, 80), dict(masked=True, jump=3e-3, periodic=(1, 0, 1))),
}


def boxes(name, monkeypatch):
    size, kw = BOXES[name]
    kw = dict(kw)
    q = kw.setdefault("q", 19)
    n = size[0] * size[1] * size[2]
    if kw.pop("masked", False):
        kw["solid"] = (O.uniform01(7, np.arange(n, dtype=np.uint64)) < 0.2).astype(np.uint8)
    kw["density_jump_x"] = kw.pop("jump", 0.0)
    gather = kw.pop("gather", False)
    if "split" in name:
        monkeypatch.setenv("LBM_DENSE_PAIR_CELLS", "2")
    f = 0.05 + 0.001 * np.random.default_rng(3).random((q, n))
    if kw.get("storage", "f64") != "f64":
        f = None
    elif "solid" in kw:
        f[:, kw["solid"] != 0] = 0.0
    lats = []
    for pair in "10":
        monkeypatch.setenv("LBM_DENSE_PAIR", pair)
        if gather and pair == "1":
            monkeypatch.setenv("LBM_DENSE_PUSH_GATHER", "1")
        lats.append(DenseLattice(*size, omega=1 / 0.8, **kw))
    return lats, f


@pytest.mark.parametrize("name", BOXES)
def test_calls_of_every_kind(name, monkeypatch):
    (a, b), f = boxes(name, monkeypatch)
    print(f"[modes] {name}", flush=True)
    own = a.graph(6)
    try:
        def same(where):
            got, want = [a.get_state(), *a.moments()], [b.get_state(), *b.moments()]
            if "jump" in name and "f32" in name:
                # What crosses the ends of the rows is stored with the jump or without, and read
                # back with it rounded to FP32 or not: half an FP32 ulp of the largest deviation
                # (0.06) and of the jump for each of the populations that meet in a readout.
                bound = 2.0 ** -24 * (0.06 + 3e-3)
                nx = BOXES[name][0][0]
                for k in range(3):
                    x, y = (v.reshape(-1, nx) if k < 2 else v.T.reshape(-1, nx) for v in (got[k], want[k]))
                    assert np.abs(x - y).max() <= bound * (1 if k == 0 else 2 * 9), where
                    assert np.array_equal(x[:, 1:-1], y[:, 1:-1]), where
            else:
                assert all(np.array_equal(x, y) for x, y in zip(got, want)), where
            m = b.mass()
            assert abs(a.mass() - m) <= 1e-12 * abs(m), where

        def restart(k):
            for lat in (a, b):
                if f is not None and k % 2 == 0:
                    lat.set_state(f)
                else:
                    lat.init_tgv(0.03, 1e-3, 5 + k)
            if f is not None and k % 2 == 0:
                assert np.array_equal(b.get_state(), f)
            same(f"start {k}")

        calls = ([1] * 4, [20], [1] * 3, [2, 2, 2, 2, 2], [1] * 5, "graph", [3], [1], [9], [1] * 4, "graph",
                 "graph", [1, 1, 1, 2, 1, 1, 1], [8], [5])
        for k in range(2):
            restart(k)
            for group in calls if k == 0 else calls[::-1]:
                for n in [0] if group == "graph" else group:
                    if group == "graph":
                        if a.info()["time_step"] % 2:
                            a.step(1)
                            b.step(1)
                        own.launch(2)
                        b.step(12)
                    else:
                        a.step(n)
                        b.step(n)
                same(f"{k} {group}")
    finally:
        if own:
            own.close()
        a.close()
        b.close()


@pytest.mark.parametrize("ones", [0, 3, 4])
@pytest.mark.parametrize("name", ["pull_walls_f64", "aa_walls_f64", "aa_jump_f64", "push_jump_f64",
                                  "pull_split_f16", "aa_f64_128"])
def test_caller_graph_in_either_mode(name, ones, monkeypatch):
    """A caller's graph captured right after a start, or after single steps."""
    (a, b), f = boxes(name, monkeypatch)
    stream, own = _Stream(), None
    print(f"[modes] caller graph {name} after {ones}", flush=True)
    try:
        a.set_stream(stream.s.value)
        for lat in (a, b):
            lat.init_tgv(0.03, 1e-3, 5)
            for _ in range(ones):
                lat.step(1)
        graph, exe = stream.capture(lambda: a.step(4))
        own = a.graph(2)
        for call in (lambda: [lat.step(2) for lat in (a, b)],
                     lambda: [lat.step(1) for lat in (a, b) for _ in range(6)],
                     lambda: [lat.step(30) for lat in (a, b)],
                     lambda: (own.launch(3), b.step(6)),
                     lambda: None if ones % 2 else [lat.init_tgv(0.02, 1e-3, 6) for lat in (a, b)],
                     lambda: [lat.step(2) for lat in (a, b)]):
            stream.launch(exe)
            b.step(4)
            call()
            stream.launch(exe)
            b.step(4)
            assert np.array_equal(a.get_state(), b.get_state())
        stream.synchronize()
        stream.destroy_graph(graph, exe)
    finally:
        if own:
            own.close()
        a.close()
        b.close()
        stream.close()
