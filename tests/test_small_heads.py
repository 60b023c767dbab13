"""Listing the heads in one workgroup (up to 5,120 particles) and in two launches,
around the workgroup's rounds of 1,024 slots and the limit.  Bitwise against the
CPU oracle."""
import numpy as np
import pytest

import oracle
from fluidsimulator_amd import hip
from tests.helpers import same_bits
from tests.test_rank_sort import cloud

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    hip.load_library()
    ok, _, err = hip.hip_device_available()
    assert ok, f"no HIP device: {err}"
    oracle.build(ref=False)


@pytest.mark.parametrize("n", [1, 1024, 1025, 4096, 4097, 5119, 5120, 5121, 8193])
@pytest.mark.parametrize("tiles", [1, 2])
def test_heads(n, tiles):
    p, pos, vel = cloud(n, 120 + n)
    pos[:, n // 2:n // 2 + n // 8] = pos[:, :1]  # a run, and a dense cell
    vel[:, n // 2:n // 2 + n // 8] = vel[:, :1]
    o = oracle.step(p, pos, vel, nsteps=2, diag="light")
    with hip.HipSolver(p, [n], tile_gather=tiles) as s:
        s.upload(pos, vel)
        s.step(2)
        r, d, pairs = s.download(), s.diag(), s.stats()["pairs"]
    assert same_bits(r.pos, o["pos"]) and same_bits(r.vel, o["vel"])
    assert np.array_equal(d["nbr_count"], o["nbr_count"])
    assert pairs == int(o["nbr_count"].astype(np.int64).sum())
