"""Runs of identical particles where every particle's list is stored (recorded
substeps, diagnostics): a run is computed once, and the lists of its slots come
from the head's row or from walks over runs.  Lists against the CPU oracle,
gradients against the gather modes that compute every particle."""
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


def points(kind):
    """Positions whose copies follow one another, or lie apart, in id order."""
    rng = np.random.default_rng(len(kind))
    if kind == "rows":      # up to 31 slots to a cell, runs of 1 to 20
        cells = np.stack(np.meshgrid(*[np.arange(4, 9)] * 3, indexing="ij")).reshape(3, -1)
        pts = []
        for c in cells.T[rng.random(125) < 0.5]:
            reps = rng.choice([1, 1, 2, 3, 4, 20], rng.integers(1, 5))
            while reps.sum() > 31:
                reps = reps[1:]
            x = 0.1 * c[:, None] + rng.uniform(0.002, 0.098, (3, len(reps)))
            pts.append(np.repeat(x, reps, 1))
        pos = np.concatenate(pts, 1)
    elif kind == "dense":   # cells of runs of up to 150 slots, and single particles
        x = 0.45 + 0.2 * rng.random((3, 120))
        pos = np.repeat(x, rng.choice([1, 1, 2, 33, 64, 65, 150], 120), 1)
    elif kind == "pile":    # most particles at three points
        x = np.array([[0.5, 0.52, 0.58]] * 3)
        pos = np.concatenate([np.repeat(x, [700, 40, 1], 1), 0.4 + 0.2 * rng.random((3, 60))], 1)
    elif kind == "apart":   # copies apart in id, so that runs end at other particles
        x = 0.45 + 0.12 * rng.random((3, 40))
        pos = np.repeat(x, 6, 1)[:, rng.permutation(240)]
    else:                   # lists too long for a row, some of them of runs
        pos = corner_cluster(230, 2, 0, seed=9)
        pos[:, 1::2] = pos[:, 0:pos.shape[1] - 1:2]
    return np.ascontiguousarray(pos.astype(np.float32))


KINDS = ["rows", "dense", "pile", "apart", "long"]


def params(planes=True):
    p = scenes.base_params((1.0, 1.0, 1.0), True)
    p.enable_vorticity = False
    if not planes:
        p.planes = []
    return p


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("cap", [0, 64])
def test_diagnostics(kind, cap):
    p, pos = params(), points(kind)
    n = pos.shape[1]
    vel = np.zeros_like(pos)
    for steps in (1, 3):
        o = oracle.step(p, pos, vel, nsteps=steps, diag=True, nbr_cap=n * n)
        with hip.HipSolver(p, [n], record_diag=True, neighbor_capacity=cap) as s:
            s.upload(pos, vel)
            s.step(steps)
            r, d, ids, st = s.download(), s.diag(), s.neighbors(), s.stats()
        assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])
        assert np.array_equal(d["nbr_count"], o["nbr_count"])
        assert same_bits(d["rho"], o["rho"]) and same_bits(d["lambda"], o["lambda"])
        assert np.array_equal(ids, o["nbr_ids"])
        assert st["pairs"] == len(ids) and st["tiles"] == 0


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("tiles", [1, 2])
def test_recordings(kind, tiles):
    p, pos = params(), points(kind)
    n = pos.shape[1]
    vel = np.zeros_like(pos)
    rng = np.random.default_rng(1)
    dx, dv = (rng.standard_normal((3, n)).astype(np.float32) for _ in range(2))
    o = oracle.step(p, pos, vel, nsteps=4, diag=True, nbr_cap=n * n)
    want = None
    for mode in (3, 1, 2):
        with hip.HipSolver(p, [n], wave_mode=mode, tile_gather=tiles, neighbor_capacity=512) as s:
            s.upload(pos, vel)
            s.forward_record(4, 2)
            r, ids, st = s.download(), s.neighbors(), s.stats()
            g = s.backward(dx, dv)
        assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"]), mode
        assert np.array_equal(ids, o["nbr_ids"]), mode
        assert st["pairs"] == len(ids) and st["tiles"] == 0
        if want is None:
            want = g
        for a, b in zip(want, g):
            assert np.array_equal(np.isnan(a), np.isnan(b)), mode
            assert same_bits(np.nan_to_num(a), np.nan_to_num(b)), mode
