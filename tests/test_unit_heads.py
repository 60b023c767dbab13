"""Dense units of one, two, four and eight heads: a batch's heads of dense cells
choose how many (one from 0, two from 4,096, four from 8,192, eight from 32,768
on).  Cells of about 48 particles, some of them copies with neighboring ids
(runs of identical slots, whose terms are added once per copy).  Bitwise
against the CPU oracle."""
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


def packed(cells, copies, seed):
    """48 particles in each of `cells` cells of a 12-wide block of cells, the
    first `copies` of them each followed by a copy."""
    rng = np.random.default_rng(seed)
    c = np.arange(cells)
    corner = 0.1 * np.stack([3 + c % 12, 3 + c // 12 % 6, 3 + c // 72])
    pos = np.repeat(corner, 48, 1) + rng.uniform(0.002, 0.098, (3, 48 * cells))
    pos = pos[:, rng.permutation(pos.shape[1])].astype(np.float32)
    pos = np.concatenate([np.repeat(pos[:, :copies], 2, 1), pos[:, copies:]], 1)
    return np.ascontiguousarray(pos)


@pytest.mark.parametrize("cells,copies", [
    (60, 0), (60, 500),      # 2,880 heads: units of one
    (120, 700),              # 5,760: two
    (300, 0), (300, 2000),   # 14,400: four
    (682, 0),                # 32,736: four, just
    (690, 0), (700, 3000),   # 33,120 and 33,600: eight
])
def test_units_bitwise(cells, copies):
    sc = scenes.dam_break(seed=cells, dims=(4, 4, 4), flags=True)
    pos = packed(cells, copies, cells + copies)
    vel = np.zeros_like(pos)
    with hip.HipSolver(sc.params, [pos.shape[1]]) as s:
        s.upload(pos, vel)
        s.step(1)
        got = s.download()
    o = oracle.step(sc.params, pos, vel, nsteps=1)
    assert same_bits(got.pos, o["pos"]) and same_bits(got.vel, o["vel"])
