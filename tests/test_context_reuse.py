"""Contexts take over the device memory and streams of destroyed ones: what a
former context left there (other sizes, a failed substep, grown tables) must
not show, also from several threads at once.  Bitwise against the CPU oracle."""
import threading

import numpy as np
import pytest

import oracle
from fluidsimulator_amd import hip, scenes
from tests.helpers import same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    hip.load_library()
    ok, _, err = hip.hip_device_available()
    assert ok, f"no HIP device: {err}"
    oracle.build(ref=False)


def expected(sc, steps):
    o = oracle.step(sc.params, sc.state.pos, sc.state.vel, nsteps=steps)
    return o["pos"], o["vel"]


def stepped(sc, steps, **kw):
    with hip.HipSolver(sc.params, [sc.state.n], **kw) as s:
        s.upload(sc.state.pos, sc.state.vel)
        s.step(steps)
        r = s.download()
    return r.pos, r.vel


@pytest.mark.parametrize("steps", [1, 3])
def test_sizes_in_turn(steps):
    cases = [scenes.dam_break(seed=40 + k, dims=d, flags=f) for k, (d, f) in enumerate(
        [((16, 16, 16), True), ((9, 7, 5), False), ((17, 16, 16), True), ((3, 2, 1), True),
         ((16, 16, 15), False), ((24, 20, 16), True)])]
    want = [expected(sc, steps) for sc in cases]
    for k in range(2 * len(cases)):
        sc, w = cases[k % len(cases)], want[k % len(cases)]
        # tables that start small grow: the next context may get the larger ones
        got = stepped(sc, steps, cell_capacity=64 if k % 3 == 0 else 0, tile_gather=k % 3)
        assert same_bits(got[0], w[0]) and same_bits(got[1], w[1]), k


def test_after_a_failed_substep():
    sc = scenes.dam_break(seed=50, dims=(10, 9, 8), flags=True)
    w = expected(sc, 2)
    bad = sc.state.pos.copy()
    bad[0, 3] = np.inf
    for _ in range(3):
        with hip.HipSolver(sc.params, [sc.state.n]) as s:
            s.upload(bad, sc.state.vel)
            with pytest.raises(hip.HipError):
                s.step(2)
        got = stepped(sc, 2)
        assert same_bits(got[0], w[0]) and same_bits(got[1], w[1])


def test_threads_with_contexts_of_their_own():
    cases = [scenes.dam_break(seed=60 + k, dims=(12 + k, 10, 8), flags=bool(k % 2))
             for k in range(4)]
    want = [expected(sc, 1) for sc in cases]
    wrong = []

    def work(k):
        for _ in range(12):
            st = cases[k].state.copy()
            hip.hip_step(cases[k].params, st)
            if not (same_bits(st.pos, want[k][0]) and same_bits(st.vel, want[k][1])):
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
