"""The library's host code when allocations, copies or synchronizations fail: a
call that fails says so, and no later call hands a kernel memory that is not
there or still in use.  Runs on the CPU over a HIP runtime without a device
(csrc/fake_hip.c), each case in a process of its own."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CELLS, NEIGHBORS = 2, 4  # status flags of a full cell table, of full lists
LONG = -3                # length of a list that is built on request


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("fake_hip")
    script = d / "versions"
    script.write_text("hip_4.2 { global: *; };\n"
                      "hip_4.3 { global: hipGraph*; hipStream*Capture; } hip_4.2;\n")
    subprocess.run([os.environ.get("CC", "gcc"), "-O1", "-shared", "-fPIC", "-w",
                    "-Wl,-soname,libamdhip64.so.7", f"-Wl,--version-script={script}",
                    os.path.join(HERE, "csrc", "fake_hip.c"), "-o",
                    str(d / "libamdhip64.so.7")], check=True)
    return str(d)


CASES = {}


def case(fn):
    CASES[fn.__name__] = fn
    return fn


class Fake:
    """The variables of the runtime, as attributes."""

    def __init__(self):
        self.__dict__["lib"] = C.CDLL("libamdhip64.so.7")
        self.lib.fake_live_bytes.restype = C.c_longlong

    def _var(self, name):
        t = {"flags": C.c_uint, "total": C.c_ulonglong, "tape_need": C.c_ulonglong}
        return t.get(name, C.c_int).in_dll(self.lib, "fake_" + name)

    def __getattr__(self, name):
        return self._var(name).value

    def __setattr__(self, name, v):
        self._var(name).value = v

    def live(self):
        return self.lib.fake_live()

    def live_bytes(self):
        return self.lib.fake_live_bytes()

    def pending_streams(self):
        return self.lib.fake_pending_streams()

    def all_streams(self):
        return self.lib.fake_all_streams()

    def fail_malloc(self, at=0, times=2):  # the library asks once more without its kept memory
        self.malloc_at, self.malloc_times = at, times

    def works(self):
        self.malloc_at, self.malloc_times = -1, 0

    def check(self):
        assert self.violations == 0, C.c_char.in_dll(self.lib, "fake_note")


def solver(**kw):
    from fluidsimulator_amd import hip, scenes

    p = scenes.base_params((1.0, 1.0, 1.0), True)
    p.enable_vorticity = False
    s = hip.HipSolver(p, [100], **kw)
    x = np.random.default_rng(0).random((3, 100), np.float32)
    s.upload(x, x)
    return s


def raises(code, fn, *a):
    from fluidsimulator_amd import hip

    try:
        fn(*a)
    except hip.HipError as e:
        assert e.code in (code if isinstance(code, tuple) else (code,)), e
        return True
    return False


@case
def growth_of_the_cell_table(fake):
    from fluidsimulator_amd import hip

    s = solver()
    s.step(1)
    for times in (2, 4, 100):  # ... also when the table of the old size is not there either
        fake.flags, fake.flags_times = CELLS, 1
        fake.fail_malloc(times=times)
        assert raises((hip.EHIP, hip.ECAPACITY), s.step, 1)
        # the last substep's cells are gone with the table
        assert s.stats()["pairs"] == 0 and raises(hip.ESTATE, s.diag)
        if times > 2:
            assert raises((hip.EHIP, hip.ECAPACITY), s.step, 1)
        fake.works()
        s.step(2)
        s.step(2, True)
        s.step_async(1)
        s.sync()
        s.stats(), s.diag()
        fake.check()
    s.close()


@case
def growth_of_the_lists(fake):
    from fluidsimulator_amd import hip

    s = solver(record_diag=True)
    s.step(1)
    for times in (2, 100):
        fake.flags, fake.flags_times = NEIGHBORS, 1
        fake.fail_malloc(times=times)
        assert raises(hip.ECAPACITY, s.step, 1)
        assert raises(hip.ESTATE, s.neighbors)
        fake.works()
        s.step(1)
        s.neighbors()
        fake.check()
    s.close()


@case
def lists_built_on_request(fake):
    from fluidsimulator_amd import hip

    s = solver(neighbor_capacity=100)
    fake.nwords = LONG
    s.step(1)
    fake.total = 1000  # more than the buffer holds
    for _ in range(2):
        fake.fail_malloc(times=2)
        assert raises(hip.EHIP, s.neighbors)
    # every list is still to be built, also those stored before one did not fit
    fake.works()
    n = fake.long_lists
    assert raises(hip.ESTATE, s.neighbors)  # (only the first is, here)
    assert fake.long_lists > n
    fake.check()
    s.step(1)
    fake.check()
    s.close()


@case
def recording(fake):
    from fluidsimulator_amd import hip

    failed = 0
    for at in range(100):
        s = solver()
        fake.fail_malloc(at=at)
        bad = raises(hip.EHIP, s.forward_record, 6, 3)
        fake.works()
        failed += bad
        if bad:
            assert raises(hip.ESTATE, s.backward)
        for steps, every in ((6, 3), (4, 2)):
            s.forward_record(steps, every)
            s.backward()
        fake.check()
        s.close()
        if not bad:
            break
    assert failed > 10
    # a tape whose lists outgrew it
    s = solver()
    s.forward_record(4, 2)
    fake.tape_need = 12345
    fake.fail_malloc()
    assert raises(hip.EHIP, s.forward_record, 4, 2)
    fake.works()
    s.forward_record(4, 2)
    s.backward()
    fake.check()
    s.close()


@case
def kept_memory_is_idle(fake):
    from fluidsimulator_amd import hip

    solver().close()
    kept, streams = fake.live(), fake.all_streams()
    assert kept > 1 and streams == 2 and fake.pending_streams() == 0
    before = fake.mallocs
    s = solver()  # takes what the first one left
    assert fake.mallocs == before and fake.all_streams() == streams
    # a context whose work may still run leaves nothing
    s.step(1)
    fake.sync_fails = 1
    s.close()
    fake.sync_fails = 0
    assert fake.live() == 1 and fake.all_streams() == 0  # (the mark of the device)
    # contexts that fail on the way: nothing that is in use is kept
    for sync_fails in (0, 1):
        for at in range(3):
            fake.copy_at, fake.sync_fails = at, sync_fails
            bad = raises(hip.EHIP, solver)
            fake.copy_at, fake.sync_fails = -1, 0
            assert bad  # the segments, the scene tables, the upload
            assert fake.pending_streams() == 0
            if sync_fails:
                assert fake.live() == 1 and fake.all_streams() == 0
    fake.check()


@case
def kept_memory_is_bounded(fake):
    from fluidsimulator_amd import hip

    solver(cell_capacity=1 << 12, neighbor_capacity=1 << 12).close()
    small = fake.live()
    # blocks larger than all that may be kept drive nothing out
    solver(cell_capacity=100 << 20, neighbor_capacity=100 << 20).close()
    assert fake.live() == small
    # ... and smaller ones the oldest only
    for k in range(20):
        s = solver(cell_capacity=(8 + k) << 20, neighbor_capacity=1 << 12)
        t = solver(cell_capacity=(4 + k) << 20, neighbor_capacity=1 << 14)
        s.close(), t.close()
        assert fake.live_bytes() <= (256 << 20) + 4099
    assert fake.live_bytes() > 100 << 20
    for k in range(40):  # ... many small ones too
        a = [solver(cell_capacity=4000 + 500 * i, neighbor_capacity=4000 + 700 * i)
             for i in range(30)]
        for s in a:
            s.close()
    assert fake.live() <= 64 + 1 and fake.all_streams() <= 8
    s = solver()
    hip.release_kept()
    s.step(1)
    assert fake.live() == 3 and fake.all_streams() == 2  # the live context's
    s.close()
    # an allocation that finds no memory gets the kept blocks'
    s = solver()
    s.close()
    fake.fail_malloc(times=1)
    s = solver(cell_capacity=1 << 26, neighbor_capacity=1 << 26)
    s.close()
    hip.release_kept()
    assert fake.live() == 0 and fake.all_streams() == 0
    solver().close()
    fake.check()


@case
def a_reset_device(fake):
    from fluidsimulator_amd import hip

    for _ in range(3):
        s = solver()
        s.step(1)
        s.close()
        fake.lib.hipDeviceReset()
        s = solver()
        s.step(1)
        s.close()
        assert fake.live() == 4 and fake.all_streams() == 2  # three blocks and the mark
    fake.lib.hipDeviceReset()
    solver().close()
    hip.release_kept()
    assert fake.live() == 0 and fake.all_streams() == 0
    fake.check()


@case
def a_stream_that_cannot_be_made(fake):
    from fluidsimulator_amd import hip

    fake.stream_fails = 1
    assert raises(hip.EHIP, solver)
    fake.stream_fails = 0
    s = solver()
    mine = C.c_void_p()
    assert fake.lib.hipStreamCreateWithFlags(C.byref(mine), 0) == 0
    for first in (None, mine):
        assert s.lib.fluid_hip_set_stream(s.h, first) == 0
        fake.stream_fails = 1
        assert s.lib.fluid_hip_set_stream(s.h, None) == hip.EHIP
        fake.stream_fails = 0
        s.step(1)
        s.download()
    assert s.lib.fluid_hip_set_stream(s.h, None) == 0
    s.step(1)
    s.close()
    assert fake.lib.hipStreamDestroy(mine) == 0
    fake.check()


@pytest.mark.parametrize("name", sorted(CASES))
def test_host_path(runtime, name):
    env = dict(os.environ, LD_LIBRARY_PATH=runtime, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), name], env=env, cwd=ROOT,
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


if __name__ == "__main__":
    f = Fake()
    CASES[sys.argv[1]](f)
    f.check()
