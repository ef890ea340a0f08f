"""A scene's state read back in several windows and with dead particles left out, and scenes in the memory of destroyed ones."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PARTICLES = ("px", "py", "vx", "vy", "pid", "particle_viscosity")


def _one(fg, scene, name, like):
    """One array of the state alone (its own offsets and windows)."""
    a = np.zeros_like(like) if name not in PARTICLES else np.zeros(scene.params.max_particles, like.dtype)
    st = fg.SceneState()
    setattr(st, name, a.ctypes.data)
    fg._check(fg.lib().fg_scene_get_state(scene.h, C.byref(st)))
    return a[:st.n_particles] if name in PARTICLES else a


WINDOW = 16 << 20


def _stream(I, J, n, visc):
    """Where the packed state's first plain array and its end lie: each component of n particles (4 bytes), then each array
    of what Scene.get_state asks for, every one on a 256-byte boundary."""
    C, U, V = I * J, (I + 1) * J, I * (J + 1)
    pad = lambda b: (b + 255) // 256 * 256  # noqa: E731
    arrays = [4 * U, 4 * V, U, V, C, 4 * C, 4 * C, 4 * C, 4 * C, 4 * U, 4 * V, 8 * C, 8 * C, C, 4 * C, 4 * U, 4 * V]
    first = pad(4 * n) * (6 if visc else 5)
    return first, first + sum(pad(b) for b in arrays + ([4 * C] if visc else []))


# One window, ragged sides, viscosity; two; five (a window is 16 MiB); the plain arrays starting 256 bytes before a window's
# end, the components filling their sections and not, and 1,024 bytes after it.  The larger ones with more particles than
# 2 ppc a cell.
@pytest.mark.parametrize("I,J,n,visc,windows,first", [
    (37, 61, 900, True, 1, None), (513, 259, 500_001, False, 2, None), (1021, 767, 1_500_000, False, 5, None),
    (523, 67, 838_848, False, 2, -256), (523, 67, 838_785, False, 2, -256), (523, 67, 838_849, False, 2, 1024)])
def test_state_arrays_and_erased_particles(fg, ctx, I, J, n, visc, windows, first):
    at, end = _stream(I, J, n, visc)
    assert (end + WINDOW - 1) // WINDOW == windows and (first is None or at - WINDOW == first), (at, end)
    rng = np.random.default_rng(I)
    walls, _ = fg.dam_break_geometry(I)
    p = fg.make_params(I, J, ppc=2, viscosity=visc, max_particles=n + 7)
    with fg.Scene(ctx, p) as sc:
        sc.init_objects(solids=[fg.box(0, p.dx, 0, J * p.dx)], friction=np.zeros(1, np.float32))
        s0 = sc.get_state()
        s0.update(px=rng.uniform(2, I - 2, n).astype(np.float32), py=rng.uniform(2, min(J - 2, 40), n).astype(np.float32),
                  vx=rng.normal(size=n).astype(np.float32), vy=rng.normal(size=n).astype(np.float32),
                  pid=rng.permutation(n).astype(np.uint32), particle_viscosity=rng.random(n).astype(np.float32))
        sc.set_state(s0)
        g = sc.get_state()
        for k in PARTICLES[:5] + (("particle_viscosity",) if visc else ()):
            assert np.array_equal(g[k], s0[k]), k
        assert np.array_equal(g["solid_sdf"], s0["solid_sdf"]) and np.array_equal(g["material"], s0["material"])
        st = sc.substep(1e-3)
        g = sc.get_state()
        assert st.particles_erased > 0 or n <= 4 * (I - 4) * (min(J - 2, 40) - 2)   # more particles than the cells may keep
        assert len(g["px"]) == sc.particle_count() == n - st.particles_killed - st.particles_erased
        # (cell, id) order, at most 2 ppc a cell, every id once
        cell = np.floor(g["px"]).astype(np.int64) * J + np.floor(g["py"]).astype(np.int64)
        assert np.all(np.diff(cell) >= 0) and np.bincount(cell).max() <= 4
        assert len(np.unique(g["pid"])) == len(g["pid"])
        same = np.diff(cell) == 0
        assert np.all(np.diff(g["pid"].astype(np.int64))[same] > 0)
        for k, a in g.items():
            if isinstance(a, np.ndarray):
                assert np.array_equal(_one(fg, sc, k, a).view(np.uint8), a.view(np.uint8)), k


def test_scene_in_pooled_memory_equals_fresh(fg):
    def frames(ctx, n, seed):
        with fg.dam_break_scene(ctx, n, ppc=4, seed=seed) as sc:
            for _ in range(2):
                sc.step_frame()
            return sc.get_state()

    with fg.Context(0) as fresh:
        want = [frames(fresh, 64, 1)]
    with fg.Context(0) as fresh:
        want.append(frames(fresh, 60, 2))
    with fg.Context(0) as ctx:
        used = ctx.bytes_in_use()
        frames(ctx, 64, 9)
        got = [frames(ctx, 64, 1), frames(ctx, 60, 2)]   # the same size, and a smaller one in the larger's memory
        assert ctx.bytes_in_use() == used
    for g, w in zip(got, want):
        for k in ("px", "py", "vx", "vy", "pid", "u", "v", "material", "fluid_sdf", "pressure"):
            assert np.array_equal(g[k], w[k]), k


def test_pool_leaves_the_budget_to_live_scenes(fg):
    small, large = fg.make_params(64, ppc=4), fg.make_params(256, ppc=4)
    need = C.c_uint64()
    fg._check(fg.lib().fg_scene_bytes(C.byref(large), C.byref(need)))
    with fg.Context(0, hbm_budget=need.value) as ctx:
        fg.Scene(ctx, small).close()
        for _ in range(2):
            with fg.Scene(ctx, large):
                assert ctx.bytes_in_use() == need.value
                with pytest.raises(fg.FgError) as e:
                    fg.Scene(ctx, small)
                assert e.value.code == fg.E_BUDGET
        fg.Scene(ctx, small).close()


def test_seeding_beyond_capacity_leaves_no_particle(fg, ctx):
    walls, fluid = fg.dam_break_geometry(64)
    with fg.Scene(ctx, fg.make_params(64, ppc=4, max_particles=1000)) as sc:
        with pytest.raises(fg.FgError) as e:
            sc.init_geometry(walls, fluid, friction=np.zeros(4, np.float32))
        assert e.value.code == fg.E_CAPACITY and sc.particle_count() == 0
        assert len(sc.get_state()["px"]) == 0
        small = [fg.box(0.5, 0.6, 0.1, 0.2)]
        sc.init_geometry(walls, small, friction=np.zeros(4, np.float32))
        assert sc.particle_count() == len(sc.get_state()["px"]) > 0
