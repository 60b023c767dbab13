"""The passes over list heads and dense units (pbf_gather.hip) where their
routes meet: a head keeps its neighbors in a row of at most 128 slots in a
batch of this size, counts at most 256 candidates one by one (beyond that by
runs), and becomes a dense unit when its neighbors do not fit the row or its
cell holds 32 particles or more.  All of it bitwise against the CPU oracle:
positions, velocities, rho, lambda, the neighbor lists in the reference's order
(lists too long for a row are built when they are asked for) and the pair
count."""
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


def corner_cluster(m, outer, copies, seed):
    """m particles within 0.04 h of a cell corner, an eighth of them in each of
    the 8 cells that meet there (so fewer than 32 per cell up to m = 248): each
    has the m - 1 others as neighbors.  `outer`: particles in each of the 56
    cells around those 8, further than h from all of the m, which makes m +
    19 outer candidates; the first `copies` particles are repeated once, bit
    for bit."""
    rng = np.random.default_rng(seed)
    eighth = np.stack(np.meshgrid([-1, 1], [-1, 1], [-1, 1], indexing="ij")).reshape(3, 8)
    signs = np.tile(eighth, (1, (m + 7) // 8))[:, :m]
    pos = [0.5 + signs * rng.uniform(0.0005, 0.0025, (3, m))]
    cells = np.stack(np.meshgrid(*[range(-2, 2)] * 3, indexing="ij")).reshape(3, -1).T
    for c in cells:
        out = (c == -2) | (c == 1)  # the axes on which the cell lies outside
        if out.any():
            u = rng.uniform(0.04, 0.096, (3, outer))  # from the inner face of the cell
            pos.append(0.5 + 0.1 * np.where(c < 0, c + 1, c)[:, None] + np.where(c < 0, -1, 1)[:, None] * u)
    pos = np.concatenate(pos, 1).astype(np.float32)
    pos[:, m - copies:m] = pos[:, :copies]
    return np.ascontiguousarray(pos[:, rng.permutation(pos.shape[1])])


@pytest.mark.parametrize("m,outer,copies", [
    (16, 0, 0),     # one round of list lanes
    (33, 0, 4),     # more than 32 neighbors, runs of two in the rows
    (128, 0, 0),    # 127 neighbors: the row has room for one more
    (129, 0, 0),    # 128: a full row
    (130, 0, 0),    # 129: dense units of one head
    (130, 0, 20),   # ... of runs
    (200, 2, 0),    # neighbors beyond the row
    (123, 7, 0),    # 256 candidates, 122 neighbors in the row
    (124, 7, 0),    # 257 candidates: counted by runs
    (124, 7, 8),    # ... of two slots
    (129, 9, 16),   # ... a full row
    (130, 9, 16),   # ... and one too many
    (264, 0, 40),   # cells of 33: dense cells
])
@pytest.mark.parametrize("flags", [False, True])
def test_routes_of_heads_bitwise(m, outer, copies, flags):
    p = scenes.base_params((1.0, 1.0, 1.0), flags)
    p.external_forces = (0.0, 0.0, 0.0)
    pos = corner_cluster(m, outer, copies, seed=m + outer)
    n = pos.shape[1]
    vel = np.zeros_like(pos)
    o = oracle.step(p, pos, vel, nsteps=1, diag=True, nbr_cap=n * n)
    with hip.HipSolver(p, [n]) as s:
        s.upload(pos, vel)
        s.step(1)
        r, d, pairs = s.download(), s.diag(), s.stats()["pairs"]
        lists = None
        if copies == 0 and m <= 248:  # dense cells and runs keep no list
            lists = s.neighbors()
    assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])
    assert same_bits(d["rho"], o["rho"]) and same_bits(d["lambda"], o["lambda"])
    assert np.array_equal(d["nbr_count"], o["nbr_count"])
    assert pairs == int(o["nbr_count"].astype(np.int64).sum())
    if lists is not None:
        assert np.array_equal(lists, o["nbr_ids"])
    # every list stored (diagnostics), as the adjoint reads them
    with hip.HipSolver(p, [n], record_diag=True) as s:
        s.upload(pos, vel)
        s.step(1)
        full, st = s.neighbors(), s.download()
    assert np.array_equal(full, o["nbr_ids"])
    assert same_bits(st.pos, o["pos"]) and same_bits(st.vel, o["vel"])


@pytest.mark.parametrize("heads", [2000, 6000, 12000])
def test_dense_units_of_one_two_and_four_heads_bitwise(heads):
    """Dense cells with `heads` runs in all, so that units hold one, two or
    four heads; run lengths of 1 to 70 slots, cells of 5 to 90 runs (units cut
    at the cells' ends), neighbors across cells."""
    rng = np.random.default_rng(heads)
    pts, left, cell = [], heads, 0
    while left > 0:
        k = int(min(left, rng.integers(5, 91)))
        c = np.array([2 * (cell % 12), cell // 144, 2 * ((cell // 12) % 12)]) * 0.1 + 0.05
        x = c[:, None] + rng.uniform(-0.045, 0.045, (3, k))
        reps = rng.choice([1, 1, 1, 2, 3, 17, 64, 65, 70], k, p=[.3, .2, .2, .1, .1, .04, .02, .02, .02])
        reps[0] += max(0, 32 - reps.sum())
        pts.append(np.repeat(x, reps, axis=1))
        left -= k
        cell += 1
    pos = np.concatenate(pts, 1).astype(np.float32)
    # a cell's copies stay consecutive in id, so each point is one run
    p = scenes.base_params((4.0, 4.0, 4.0), True)
    p.external_forces = (0.0, 0.0, 0.0)
    p.planes = []
    vel = np.zeros_like(pos)
    n = pos.shape[1]
    print(f"{n} particles, {heads} heads in {cell} dense cells", flush=True)
    oracle.set_threads(8)
    o = oracle.step(p, pos, vel, nsteps=1, diag="light")
    with hip.HipSolver(p, [n], tile_gather=2) as s:
        s.upload(pos, vel)
        s.step(1)
        r, d, pairs = s.download(), s.diag(), s.stats()["pairs"]
    assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])
    assert same_bits(d["rho"], o["rho"])
    assert np.array_equal(d["nbr_count"], o["nbr_count"])
    assert pairs == int(o["nbr_count"].astype(np.int64).sum())
