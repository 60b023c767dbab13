"""Queries of a context describe the last substep that ran, whatever the context
was told since: other parameters, the autotuner's trials and the state it puts
back, a recorded rollout, a graph's replay of an older configuration."""
import numpy as np
import pytest

import oracle
from fluidsimulator_amd import hip, scenes
from tests.helpers import same_bits
from tests.test_gather_heads import corner_cluster

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    hip.load_library()
    ok, _, err = hip.hip_device_available()
    assert ok, f"no HIP device: {err}"
    oracle.build(ref=False)


def want(p, pos, vel, steps):
    """What the oracle has in substep `steps` (the diagnostics are its last one's)."""
    return oracle.step(p, pos, vel, nsteps=steps, diag=True, nbr_cap=400 * pos.shape[1])


def check(s, o, neighbors=True, lam=True):
    d = s.diag()
    assert np.array_equal(d["nbr_count"], o["nbr_count"])
    assert same_bits(d["rho"], o["rho"])
    if lam:
        assert same_bits(d["lambda"], o["lambda"])
    assert s.stats()["pairs"] == int(o["nbr_count"].astype(np.int64).sum())
    if neighbors:
        assert np.array_equal(s.neighbors(), o["nbr_ids"])


@pytest.fixture(scope="module")
def block():
    sc = scenes.dam_break(seed=90, dims=(14, 13, 12), flags=True)
    sc.params.enable_vorticity = False
    return sc.params, sc.state.pos, sc.state.vel


@pytest.mark.parametrize("tiles", [1, 2])
def test_other_parameters(block, tiles):
    p, pos, vel = block
    o = want(p, pos, vel, 1)
    q = scenes.dam_break(seed=90, dims=(2, 2, 2), flags=True).params
    q.h, q.solver_iterations = 0.2, 3
    with hip.HipSolver(p, [pos.shape[1]], tile_gather=tiles) as s:
        s.upload(pos, vel)
        s.step(1)
        s.set_params(q)
        check(s, o)


def test_other_parameters_and_lists_too_long_for_a_row():
    p = scenes.base_params((1.0, 1.0, 1.0), False)
    p.external_forces = (0.0, 0.0, 0.0)
    pos = corner_cluster(200, 2, 0, seed=5)
    o = want(p, pos, np.zeros_like(pos), 1)
    q = scenes.base_params((1.0, 1.0, 1.0), False)
    q.h = 0.05
    with hip.HipSolver(p, [pos.shape[1]]) as s:
        s.upload(pos, np.zeros_like(pos))
        s.step(1)
        s.set_params(q)
        check(s, o)


@pytest.mark.parametrize("tiles", [1, 2])
@pytest.mark.parametrize("knobs", [hip.TUNE_TILES, hip.TUNE_TILES | hip.TUNE_WAVE_MODE,
                                   hip.TUNE_BRICK | hip.TUNE_BLOCK])
def test_after_the_autotuner(block, tiles, knobs):
    p, pos, vel = block
    o = want(p, pos, vel, 4)  # two substeps before the trials of two each
    with hip.HipSolver(p, [pos.shape[1]], tile_gather=tiles) as s:
        s.upload(pos, vel)
        s.step(2)
        s.autotune(trial_steps=2, knobs=knobs)
        check(s, o)  # the last trial's last substep
        s.step(2)
        check(s, o)
        r = s.download()
    assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])


@pytest.mark.parametrize("tiles", [1, 2])
def test_recorded_substeps_and_replays(block, tiles):
    p, pos, vel = block
    n = pos.shape[1]
    with hip.HipSolver(p, [n], tile_gather=tiles) as s:
        s.upload(pos, vel)
        s.step(2, graph=True)
        check(s, want(p, pos, vel, 2))
        s.forward_record(3, 1)
        # (the iterates of a recorded substep are on its tape)
        check(s, want(p, pos, vel, 5), lam=False)
        s.step(1, graph=True)
        check(s, want(p, pos, vel, 6))
        s.forward_record(3, 1)
        s.backward(np.ones((3, n), np.float32), np.ones((3, n), np.float32))
        # the reverse pass ran the recording's first substep again, last
        check(s, want(p, pos, vel, 7), lam=False)
        s.step(1)
        # (the first cells of 32 particles or more, which keep no lists)
        check(s, want(p, pos, vel, 10), neighbors=False)


@pytest.mark.parametrize("tiles", [0, 1, 2])
@pytest.mark.parametrize("knobs", [hip.TUNE_BLOCK, hip.TUNE_BLOCK | hip.TUNE_TILES])
def test_the_tuner_leaves_the_tile_mode_unless_asked(tiles, knobs):
    sc = scenes.dam_break(seed=91, dims=(38, 34, 31), flags=True)  # 40,052 particles: none by default
    with hip.HipSolver(sc.params, [sc.state.n], tile_gather=tiles) as s:
        s.upload(sc.state.pos, sc.state.vel)
        rep = s.autotune(trial_steps=1, knobs=knobs)
        s.step(1)
        st = s.stats()
    assert rep["candidates_rejected"] == 0
    assert (st["tiles"] > 0) == (rep["tile_gather"] == 1)
    if knobs == hip.TUNE_BLOCK:
        assert rep["tile_gather"] == tiles
    else:
        assert rep["tile_gather"] in (1, 2)
