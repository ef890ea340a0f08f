"""The library's host code over a stand-in for the HIP runtime (hip_host_stub.cpp): what waits for what, whose memory counts
where, and which kernels a rule picks.  Each scenario runs in a process of its own, with the stand-in's symbols ahead of the runtime's."""
import ctypes as C
import os
import random
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


def _need(fg, params):
    n = C.c_uint64()
    fg._check(fg.lib().fg_scene_bytes(C.byref(params), C.byref(n)))
    return n.value


def pool_keeps_the_budget(fg, stub):
    """Scenes made and destroyed in turn, their sizes close enough that one could live in another's memory: the device
    memory stays within the budget, and what fits the budget is not refused."""
    rng = random.Random(5)
    sizes = {n: _need(fg, fg.make_params(n, ppc=4)) for n in (32, 40, 48, 56, 60, 62, 64)}
    budget = 5 * sizes[64]
    with fg.Context(0, hbm_budget=budget) as ctx:
        base, live, refused = stub.stub_device_bytes(), [], 0
        for step in range(600):
            n = rng.choice(list(sizes))
            if rng.random() < 0.45 and live:
                live.pop(rng.randrange(len(live)))[0].close()
            else:
                held = sum(b for _, b in live)
                try:
                    live.append((fg.Scene(ctx, fg.make_params(n, ppc=4)), sizes[n]))
                except fg.FgError as e:
                    assert e.code == fg.E_BUDGET and held + sizes[n] > budget, (step, held, sizes[n])
                    refused += 1
            assert ctx.bytes_in_use() == sum(b for _, b in live), step
            # the arenas; a descriptor of a few KB a block lies beside each
            assert stub.stub_device_bytes() - base <= budget + 64 * 4096, (step, stub.stub_device_bytes() - base, budget)
        assert refused > 20
        for sc, _ in live:
            sc.close()


def server_keeps_its_budget(fg, stub):
    """A server's budget bounds the device memory of its scenes and of the memory kept from those that ended, on a context
    that has no budget of its own and whose own scenes left memory in the pool."""
    rng = random.Random(7)
    walls, fluids = fg.dam_break_geometry(32)
    with fg.Context(0) as ctx:
        base = stub.stub_device_bytes()
        for sc in [fg.Scene(ctx, fg.make_params(64, ppc=4)) for _ in range(12)]:
            sc.close()
        largest = _need(fg, fg.make_params(96, ppc=4))
        with fg.Server(ctx, hbm_budget=3 * largest, max_resident=16) as srv:
            kept, waits = [], 0
            for tick in range(200):
                for _ in range(rng.randint(0, 3)):
                    n, keep = rng.choice((40, 56, 64, 72, 88, 90, 96)), rng.random() < 0.3
                    p = fg.make_params(n, ppc=4)
                    rid = srv.submit(p, walls, fluids, rng.randint(1, 4), keep=keep)
                    if keep:
                        kept.append(rid)
                t = srv.tick()
                waits += t.queued > 0
                held = stub.stub_device_bytes() - base
                # beside the scenes: the lane's descriptors and block maps
                assert held <= 3 * largest + (1 << 20), (tick, held, 3 * largest)
                if kept and rng.random() < 0.3 and srv.status(kept[0]).state == fg.REQ_DONE:
                    srv.release(kept.pop(0))
            assert waits > 20


def pool_gives_way_to_every_allocation(fg, stub):
    """Where the device has no memory left, what destroyed scenes left behind is given back: to a batch's buffers (on each
    lane's own thread), to a set-up's polygons, to a probe, to another context and its scenes."""
    walls, fluids = fg.dam_break_geometry(32)
    many = [fg.box(0.2 + 1e-3 * k, 0.21 + 1e-3 * k, 0.1, 0.3) for k in range(600)]

    def batch(ctx, lanes):
        scenes = [fg.Scene(ctx, fg.make_params(32, ppc=4)) for _ in range(8)]
        ctx.set_batch_lanes(lanes)
        return scenes, lambda: fg.batch_step_frame(ctx, scenes)

    def setup(ctx):
        scenes = [fg.Scene(ctx, fg.make_params(32, ppc=4))]
        return scenes, lambda: scenes[0].init_geometry(walls, many)

    def other(ctx):
        def call():
            with fg.Context(0) as second, fg.Scene(second, fg.make_params(48, ppc=4)) as sc:
                sc.init_geometry(walls, fluids)
        return [], call

    def probe(ctx):
        return [], lambda: ctx.bandwidth_probe(4 << 20, 1)

    def scene(ctx):
        return [], lambda: fg.Scene(ctx, fg.make_params(96, 64, ppc=4)).close()

    for make in (lambda c: batch(c, 1), lambda c: batch(c, 4), setup, other, probe, scene):
        with fg.Context(0) as ctx:
            live, call = make(ctx)
            for sc in [fg.Scene(ctx, fg.make_params(64, ppc=4)) for _ in range(12)]:
                sc.close()
            stub.stub_limit(stub.stub_device_bytes())   # not a byte beyond what is held
            call()
            stub.stub_limit(2**63)
            for sc in live:
                sc.close()


def _batch(fg, ctx, sizes):
    out = []
    for n in sizes:
        walls, fluids = fg.dam_break_geometry(n)
        out.append(fg.Scene(ctx, fg.make_params(n, ppc=1)))
        out[-1].init_geometry(walls, fluids)
    return out


def sdf_lanes_by_the_bins_of_the_group(fg, stub):
    """k_sdf_materials' 32 lanes a bin where the bins of the group's scenes together are few, however uneven their sizes."""
    for sizes, few in (([64] * 8, True), ([256] + [32] * 40, True), ([256] * 4, False), ([512] + [32], False), ([32] * 250, False)):
        with fg.Context(0) as ctx:
            scenes = _batch(fg, ctx, sizes)
            stub.stub_reset_launches()
            fg.batch_step_frame(ctx, scenes)
            wide, plain = (stub.stub_launches(b"k_sdf_materialsILi%dE" % k) for k in (32, 4))
            assert (wide > 0, plain > 0) == (few, not few), (sizes[0], len(sizes), wide, plain)
            for sc in scenes:
                sc.close()


def bands_polled_where_empty_ones_cost_more(fg, stub):
    """A level set of nine bands at most (128^2): a few scenes launch all nine, many look after eight whether any is left
    (none is here); more than about ten bands are always looked at."""
    for count, n, want in ((1, 128, 9), (32, 128, 9), (96, 128, 8), (1, 512, 8)):
        with fg.Context(0) as ctx:
            scenes = _batch(fg, ctx, [n] * count)
            stub.stub_reset_launches()
            fg.batch_step_frame(ctx, scenes)
            got = stub.stub_launches(b"k_levelset_band")
            assert got == want, (count, n, got, want)
            for sc in scenes:
                sc.close()


SCENARIOS = [failed_launch_leaves_no_lane_busy, pool_keeps_the_budget, server_keeps_its_budget,
             pool_gives_way_to_every_allocation, sdf_lanes_by_the_bins_of_the_group,
             bands_polled_where_empty_ones_cost_more]


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
    _stub.stub_launches.argtypes = [C.c_char_p]
    _stub.stub_launches.restype = C.c_long
    _stub.stub_fail_launch.argtypes = [C.c_long]
    sys.path.insert(0, os.path.dirname(HERE))
    import flipsolver2d_amd as _fg

    next(f for f in SCENARIOS if f.__name__ == sys.argv[2])(_fg, _stub)
    assert _stub.stub_allocations() == 0
