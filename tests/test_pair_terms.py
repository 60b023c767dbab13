"""The passes' pair terms in every form they are compiled in: the tensile
correction off, with an exponent of 2, 3 or 4, through LDS tiles and without,
and lengths so small that the terms take the general form (min_r^2 below
2^-96, where the square root's short form does not hold).  Bitwise against the
CPU oracle (a NaN at the same places)."""
import numpy as np
import pytest

import oracle
from fluidsimulator_amd import hip, scenes
from tests.helpers import same_bits, same_bits_or_nan

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle():
    oracle.build(ref=False)


def step(p, pos, vel, tiles, nsteps):
    with hip.HipSolver(p, [pos.shape[1]], tile_gather=tiles) as s:
        s.upload(pos, vel)
        s.step(nsteps)
        return s.download(), s.stats()["tiles"]


@pytest.mark.parametrize("tiles", [1, 2])
@pytest.mark.parametrize("n", [0, 2, 3, 4])
def test_corrections_bitwise(n, tiles):
    p = scenes.base_params((2.0, 2.0, 2.0), True)
    p.enable_scorr = n > 0
    p.scorr_n = max(n, 2)
    pos = scenes.lattice_block(11, 9, 7, d=0.045, seed=n, jitter=0.6)
    vel = np.zeros_like(pos)
    o = oracle.step(p, pos, vel, nsteps=3)
    r, t = step(p, pos, vel, tiles, 3)
    assert (t > 0) == (tiles == 1)
    assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])


@pytest.mark.parametrize("h", [1.0, 2.0 ** -20, 2.0 ** -44])
def test_general_form_bitwise(h):
    """Positions in units of h: at 2^-44 the terms are of the general form and
    no brick is a tile."""
    p = scenes.base_params((2.0, 2.0, 2.0), True)
    p.planes = []
    p.external_forces = (0.0, 0.0, 0.0)
    p.h = float(np.float32(h))
    pos = (scenes.lattice_block(9, 8, 7, d=0.45, seed=3, jitter=0.6) * np.float32(h)).astype(np.float32)
    pos[:, 40] = pos[:, 41]  # a pair closer than min_r
    vel = np.zeros_like(pos)
    o = oracle.step(p, pos, vel, nsteps=1)
    for tiles in (1, 2):
        r, t = step(p, pos, vel, tiles, 1)
        assert (t > 0) == (tiles == 1 and h > 2.0 ** -40)
        assert same_bits_or_nan(r.pos, o["pos"]) and same_bits_or_nan(r.vel, o["vel"])
