"""The library's host code over a stand-in for the HIP runtime (hip_host_stub.cpp): what waits for what, and whose memory
counts where.  Each scenario runs in a process of its own, with the stand-in's symbols ahead of the runtime's."""
import ctypes as C
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _viscous(fg, ctx, n):
    walls, fluids = fg.dam_break_geometry(n)
    sc = fg.Scene(ctx, fg.make_params(n, ppc=4, viscosity=True))
    sc.init_geometry(walls, fluids)
    return sc


def failed_launch_leaves_no_lane_busy(fg, stub):
    """A destroyed scene's memory goes to the next scene, so nothing may be queued on it any more: also where a step
    failed on a lane other than the first."""
    failures = 0
    for launch in range(0, 400, 7):
        with fg.Context(0) as ctx:
            scenes = [_viscous(fg, ctx, n) for n in (64, 48, 40, 32)]
            ctx.set_batch_lanes(2)
            stub.stub_fail_launch(launch)
            try:
                fg.batch_step_frame(ctx, scenes)
                assert not stub.stub_launch_failed()
            except fg.FgError as e:
                assert e.code == fg.E_DEVICE
                failures += 1
            for sc in scenes:
                sc.close()
            busy = stub.stub_busy_streams()
            stub.stub_fail_launch(-1)
            assert busy == 0, (launch, busy)
    assert failures > 10


SCENARIOS = [failed_launch_leaves_no_lane_busy]


@pytest.fixture(scope="module")
def stub_lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libhiphoststub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall", os.path.join(HERE, "hip_host_stub.cpp"), "-o", out],
                   check=True)
    return out


@pytest.mark.parametrize("scenario", [f.__name__ for f in SCENARIOS])
def test_host(stub_lib, scenario):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub_lib, scenario], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    _stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    _stub.stub_device_bytes.restype = _stub.stub_allocations.restype = C.c_uint64
    _stub.stub_limit.argtypes = [C.c_uint64]
    _stub.stub_fail_launch.argtypes = [C.c_long]
    sys.path.insert(0, os.path.dirname(HERE))
    import flipsolver2d_amd as _fg

    next(f for f in SCENARIOS if f.__name__ == sys.argv[2])(_fg, _stub)
    assert _stub.stub_allocations() == 0
