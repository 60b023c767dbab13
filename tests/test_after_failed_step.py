"""What a context tells about its neighbors after a substep that failed: the
grid, slots and lists are still those of the last good substep, the statistics
count no pairs, lists that would have to be built are refused, and the state
is the last committed one."""
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


def scene(kind):
    """Particles with dense cells, or with lists too long for a row (or neither),
    and one that flies off to the right at 600 units a second."""
    rng = np.random.default_rng(7)
    if kind == "dense":  # cells of up to 80 particles
        pos = rng.uniform(0.2, 0.6, (3, 3000)).astype(np.float32)
    elif kind == "long":
        pos = corner_cluster(200, 2, 0, seed=1)
    else:
        pos = scenes.dam_break(seed=8, dims=(12, 11, 10), flags=True).state.pos
    pos = np.concatenate([pos, np.full((3, 1), 0.9, np.float32)], 1)
    vel = np.zeros_like(pos)
    vel[0, -1] = 600.0
    p = scenes.base_params((4.0, 4.0, 4.0), True)
    p.external_forces = (0.0, 0.0, 0.0)
    p.planes = []
    return p, np.ascontiguousarray(pos), vel


def queries(s, kind):
    """Every query of a context; the statistics."""
    st = s.stats()
    d = s.diag()
    assert sorted(d["sorted_ids"]) == list(range(s.n))
    try:
        ids = s.neighbors()
        assert ids.min(initial=0) >= 0 and ids.max(initial=0) < s.n
    except hip.HipError as e:
        assert e.code == hip.ESTATE
        assert kind != "plain"
    return st


@pytest.mark.parametrize("kind", ["plain", "dense", "long"])
@pytest.mark.parametrize("tiles", [0, 1])
@pytest.mark.parametrize("how", ["range", "cells"])
def test_queries_after_a_failed_substep(kind, tiles, how):
    p, pos, vel = scene(kind)
    n = pos.shape[1]
    o = oracle.step(p, pos, vel, nsteps=1, diag="light")
    # the table of the first substep has room, that of a later one has not
    cap = 1 << 16 if how == "cells" else 0
    with hip.HipSolver(p, [n], cell_capacity=cap, tile_gather=tiles) as s:
        s.upload(pos, vel)
        s.step(1)
        keys, before = s.grid()
        assert s.stats()["pairs"] == int(o["nbr_count"].astype(np.int64).sum())
        if how == "range":
            q = scenes.base_params((4.0, 4.0, 4.0), True)
            q.planes = []
            q.external_forces = (0.0, 3e38, 0.0)
            s.set_params(q)
            with pytest.raises(hip.HipError) as e:
                s.step(2)
            assert e.value.code == hip.ERANGE
        else:
            s.step_async(200)
            with pytest.raises(hip.HipError) as e:
                s.sync()
            assert e.value.code == hip.ECAPACITY
        r = s.download()
        if how == "range":
            assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])
            _, after = s.grid()
            assert np.array_equal(before, after)
        assert np.isfinite(r.pos).all()
        # dense cells keep no lists: nothing is counted for a failed substep
        assert queries(s, kind)["pairs"] == 0
        # ... and the context is as good as new
        s.set_params(p)
        s.upload(pos, vel)
        s.step(1)
        r = s.download()
        assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])
        assert s.stats()["pairs"] == int(o["nbr_count"].astype(np.int64).sum())


@pytest.mark.parametrize("edge", [1, 2, 4, 8])
@pytest.mark.parametrize("count", [1, 2, 40])
def test_scenes_over_the_whole_coordinate_range_do_not_fit(edge, count):
    """Particles at opposite corners of the range of cell coordinates: the cells
    of the table, in one scene or in all, exceed 64 bits."""
    p = scenes.base_params((4.0, 4.0, 4.0), False)
    p.planes = []
    p.external_forces = (0.0, 0.0, 0.0)
    end = 0.0999999 * (1 << 20)
    pos = np.tile(np.array([[-end, end]] * 3, np.float32), (1, count))
    with hip.HipSolver([p] * count, [2] * count, brick_edge=edge) as s:
        s.upload(pos, np.zeros_like(pos))
        with pytest.raises(hip.HipError) as e:
            s.step(1)
        assert e.value.code == hip.ECAPACITY
        assert same_bits(s.download().pos, pos)


@pytest.mark.parametrize("count", [17, 65, 1024, 1025, 2100])
def test_grids_of_many_scenes(count):
    """Scenes beyond the threads of the grid setup, some of them empty: bitwise,
    also after a substep whose table did not fit and after one that had a
    particle out of range."""
    p = scenes.base_params((4.0, 4.0, 4.0), True)
    p.planes = []
    rng = np.random.default_rng(count)
    counts = [0 if k % 7 == 3 else int(rng.integers(1, 9)) for k in range(count)]
    n = sum(counts)
    pos = (0.2 + 0.3 * rng.random((3, n))).astype(np.float32)
    vel = rng.standard_normal((3, n)).astype(np.float32)
    want, at = [], 0
    for c in counts:
        if c:
            o = oracle.step(p, pos[:, at:at + c], vel[:, at:at + c], nsteps=2)
            want.append(np.concatenate([o["pos"], o["vel"]]))
        at += c
    want = np.concatenate(want, 1)
    with hip.HipSolver([p] * count, counts, cell_capacity=1000) as s:
        s.upload(pos, vel)
        s.step(1)
        _, grid = s.grid()
        assert (grid[:, 7] > 0).sum() == sum(c > 0 for c in counts)
        assert np.array_equal(grid[:, 6], np.concatenate([[0], np.cumsum(grid[:-1, 7])]))
        s.step(1)
        r = s.download()
        assert same_bits(np.concatenate([r.pos, r.vel]), want)
        _, grid = s.grid()
        q = scenes.base_params((4.0, 4.0, 4.0), True)
        q.planes, q.external_forces = [], (0.0, 0.0, 3e38)
        s.set_params(q)
        with pytest.raises(hip.HipError):
            s.step(1)
        assert np.array_equal(s.grid()[1], grid)
        s.set_params(p)
        s.upload(pos, vel)
        s.step(2)
        r = s.download()
        assert same_bits(np.concatenate([r.pos, r.vel]), want)
