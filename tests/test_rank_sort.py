"""The sort of small batches by counting (one launch up to 8,192 particles, the
radix sort beyond): blocks of 32 ids, the last one ragged, several workgroups
per cell, scenes of a batch that share a block.  After the first substep the
slots are no longer in id order.  Bitwise against the CPU oracle."""
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


def cloud(n, seed):
    """n particles at random places of a box (about 8 per cell, ids in no
    order); the params of a dam break."""
    rng = np.random.default_rng(seed)
    sc = scenes.dam_break(seed=seed, dims=(4, 4, 4), flags=True)
    edge = max(0.1, 0.05 * n ** (1.0 / 3.0))
    pos = (0.3 + edge * rng.random((3, n))).astype(np.float32)
    vel = rng.standard_normal((3, n)).astype(np.float32)
    return sc.params, pos, vel


def check(parts, steps):
    with hip.HipSolver([p for p, _, _ in parts], [x.shape[1] for _, x, _ in parts]) as s:
        s.upload(np.concatenate([x for _, x, _ in parts], 1),
                 np.concatenate([v for _, _, v in parts], 1))
        s.step(steps)
        got = s.download()
    at = 0
    for p, x, v in parts:
        o = oracle.step(p, x, v, nsteps=steps)
        b = at + x.shape[1]
        assert same_bits(got.pos[:, at:b], o["pos"]) and same_bits(got.vel[:, at:b], o["vel"])
        at = b


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 64, 65, 1023, 1024, 1025, 8161, 8191, 8192, 8193])
def test_one_scene(n):
    check([cloud(n, 70 + n)], 3)


@pytest.mark.parametrize("sizes", [(1, 31, 1), (33, 5, 100, 2), (4000, 17, 4175), (4000, 17, 4176)])
def test_scenes_of_a_batch(sizes):
    check([cloud(n, 90 + k) for k, n in enumerate(sizes)], 3)


def test_one_cell_holds_all():
    p, pos, vel = cloud(1500, 5)
    pos = np.full_like(pos, 0.55)
    pos[0] += np.linspace(0.0, 0.03, pos.shape[1], dtype=np.float32)[::-1]
    check([(p, np.ascontiguousarray(pos), np.zeros_like(vel))], 2)
