"""The lists of a recorded substep, copied from the list heads' rows by
workgroups that take consecutive heads (k_store_rows): more than 32 heads to a
workgroup, a last workgroup with few, and scenes that end inside one.  The
gradients of a batch of equal scenes are, bit for bit, those of the one scene
on its own, whose workgroups take at most 32 heads each."""
import numpy as np
import pytest

from fluidsimulator_amd import hip, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies,dims", [(1, (3, 1, 1)), (33, (16, 9, 7)), (40, (11, 10, 9)),
                                         (5, (30, 25, 18))])
def test_recorded_lists_of_many_heads(copies, dims):
    p = scenes.base_params((4.0, 3.0, 2.0), True)
    p.enable_vorticity = False
    pos = scenes.lattice_block(*dims, d=0.05, seed=11)
    n = pos.shape[1]
    vel = scenes.normal(11, 3 * n, stream=7, sigma=0.3).reshape(3, n).astype(np.float32)
    seed = np.random.default_rng(2).standard_normal((3, n)).astype(np.float32)
    print(f"{copies} scenes of {n}", flush=True)

    def gradients(k):
        with hip.HipSolver([p] * k, [n] * k, tile_gather=2) as s:
            s.upload(np.tile(pos, (1, k)), np.tile(vel, (1, k)))
            s.forward_record(3, 2)
            return s.backward(np.tile(seed, (1, k)), None)

    ex, ev, eg = gradients(1)
    dx, dv, dg = gradients(copies)
    for k in range(copies):
        sl = slice(k * n, (k + 1) * n)
        assert np.array_equal(dx[:, sl].view(np.uint32), ex.view(np.uint32)), k
        assert np.array_equal(dv[:, sl].view(np.uint32), ev.view(np.uint32)), k
        assert np.array_equal(dg[k].view(np.uint32), eg[0].view(np.uint32)), k
