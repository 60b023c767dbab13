"""Boxes and grid set up in one launch (k_predict_setup, batches of up to 32,768
particles in up to 16 scenes): the workgroup that finishes last reads boxes and
flags that other workgroups' wavefronts wrote with atomics."""
import os
import re
import subprocess

import numpy as np
import pytest

import oracle
from fluidsimulator_amd import build, hip, scenes
from tests.helpers import same_bits


def test_every_box_atomic_is_waited_for_before_the_count(tmp_path):
    """In the compiled kernel, a wavefront that has issued an atomic on a box or
    on the flags waits for it before the next barrier (which waits for none)."""
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    asm = tmp_path / "k.s"
    subprocess.run([cc, *build.HIPCC_FLAGS, "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, "pbf_kernels.hip"), "-o", str(asm)], check=True)
    text = asm.read_text()
    body = re.search(r"^_ZN\S*k_predict_setup\S*:(.*?)^\s*s_endpgm", text, re.S | re.M).group(1)
    # up to the counter, the only atomic add of the boxes' part
    body = body[:body.index("global_atomic_add")]
    pending, atomics = False, 0
    for line in body.splitlines():
        line = line.strip()
        if re.match(r"(global|flat)_atomic_(or|smin|smax)", line):
            pending, atomics = True, atomics + 1
        elif re.match(r"s_waitcnt vmcnt\(0\)", line):
            pending = False
        elif line.startswith("s_barrier"):
            assert not pending
    assert atomics == 7 and not pending


@pytest.fixture(scope="module")
def device():
    hip.load_library()
    ok, _, err = hip.hip_device_available()
    assert ok, f"no HIP device: {err}"
    oracle.build(ref=False)


def blocks(counts, seed):
    """One scene per count: the particle farthest from the others, which alone
    sets a face of its scene's box, is the first or the last of the scene, so it
    lies in whichever wavefront of a shared workgroup the scenes meet in."""
    rng = np.random.default_rng(seed)
    out = []
    for k, n in enumerate(counts):
        pos = rng.uniform(0.3, 0.9, (3, n))
        pos[:, 0] = 0.05
        pos[:, -1] = 1.5 + 0.25 * k
        out.append(np.ascontiguousarray(pos.astype(np.float32)))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("counts,block", [
    ((1920,) * 4, 256),                       # 7.5 workgroups a scene
    ((70, 130, 200, 331, 64, 65, 1, 517), 256),
    ((900, 333, 1200, 77), 1024),             # several scenes to a workgroup
    ((97,) * 16, 64),
])
@pytest.mark.parametrize("graph", [False, True])
def test_scenes_that_meet_in_a_workgroup(device, counts, block, graph):
    p = scenes.base_params((6.0, 6.0, 6.0), True)
    pos = blocks(counts, seed=sum(counts))
    steps = 24
    with hip.HipSolver([p] * len(counts), list(counts), block_size=block) as s:
        both = np.concatenate(pos, 1)
        s.upload(both, np.zeros_like(both))
        s.step(steps, graph=graph)
        r = s.download()
    at = 0
    for x in pos:
        n = x.shape[1]
        o = oracle.step(p, x, np.zeros_like(x), nsteps=steps)
        assert same_bits(r.pos[:, at:at + n], o["pos"]), at
        assert same_bits(r.vel[:, at:at + n], o["vel"]), at
        at += n


@pytest.mark.gpu
@pytest.mark.parametrize("lane", [0, 64, 200, 255, 1919])
def test_a_failed_substep_is_not_counted(device, lane):
    """The range flag of any wavefront reaches the grid setup of its substep."""
    p = scenes.base_params((6.0, 6.0, 6.0), True)
    pos = np.concatenate(blocks((1920,) * 4, seed=3), 1)
    pos[1, 1920 + lane] = np.nan
    with hip.HipSolver([p] * 4, [1920] * 4) as s:
        s.upload(pos, np.zeros_like(pos))
        for _ in range(8):
            with pytest.raises(hip.HipError) as e:
                s.step(2)
            assert e.value.code == hip.ERANGE
            assert s.download().time == 0.0
