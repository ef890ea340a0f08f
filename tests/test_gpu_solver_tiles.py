"""The solver kernels that work in tiles, where a tile can go wrong: sides of one cell more or less than a tile, grids
of one tile's width, several tiles a block; against the oracle's converged solve, and the viscosity solve's tiles."""
import ctypes as C

import numpy as np
import pytest
from helpers import oracle_state_dict, rel_l2, run_oracle_frames
from test_gpu_mg import _oracle_solve, _tank

pytestmark = pytest.mark.gpu


# The solve stops at a residual of 1e-10 ||b||; the condition of a Dirichlet 5-point matrix of n cells a side is at most
# 4 n^2 / pi^2 (3.7e4 at 300), so x is within 4e-6 of the oracle's.
@pytest.mark.parametrize("shape", [(33, 65), (31, 33), (4, 300), (300, 4), (97, 129)])
@pytest.mark.parametrize("chunk", [1024, 4096])
def test_pressure_tiles(fg, orc, ctx, shape, chunk):
    mat, b = _tank(*shape, seed=sum(shape))
    try:
        ctx.set_solver_tiling(1024 if chunk == 1024 else 2, chunk)   # two blocks: several tiles each
        x, st = ctx.poisson_solve(mat, 1.0, b, tol=1e-10)
    finally:
        ctx.set_solver_tiling()
    assert st.converged
    assert rel_l2(x, _oracle_solve(orc, mat, 1.0, b)) <= 1e-5


# The bar of the square grids: the same particles, pressure and velocities within 1e-5 (the viscosity CG stops at 1e-12).
@pytest.mark.parametrize("n_i,n_j", [(33, 47), (17, 70), (65, 31)])
def test_viscosity_tiles(fg, orc, ctx, n_i, n_j):
    dx = 1.0 / max(n_i, n_j)
    w, h = n_i * dx, n_j * dx
    walls = [fg.box(0, dx, 0, h), fg.box(w - dx, w, 0, h), fg.box(0, w, 0, dx), fg.box(0, w, h - dx, h)]
    fluids = [fg.box(0.3 * w, w - dx, dx, 0.6 * h)]
    p = orc.make_params(n_i, n_j, dx=dx, ppc=4, tol=1e-12, viscosity=True, fluid_viscosity=[2.0])
    st = orc.init_scene_objects(p, solids=walls, fluids=fluids, seed=9)
    run_oracle_frames(orc, p, st, 2)
    dt = np.float32(1.0 / 60)
    with fg.Scene(ctx, fg.make_params(n_i, n_j, dx=dx, ppc=4, tol=1e-10, viscosity=True)) as sc:
        sc.set_friction(np.zeros(4, np.float32))
        sc.set_state(oracle_state_dict(st))
        gs = sc.substep(float(dt))
        g = sc.get_state()
    orc.lib().orc_substep(C.byref(p), st.ref(), C.c_float(dt), C.byref(orc.OrcStats()))
    assert gs.converged and gs.viscosity_iters > 0
    assert np.array_equal(g["pid"], st.pid[:st.n])
    assert np.array_equal(g["viscosity"].view(np.uint32), st.viscosity.view(np.uint32))
    e = [rel_l2(g[k], getattr(st, k)) for k in ("pressure", "u", "v")]
    assert max(e) <= 1e-5, e


# A caller's own rows: counts up to the 7 that the three bits hold (materials give 4 at most), one to three above the row's
# neighbours.  The matrix is diagonally dominant by 1 and its norm at most 7 + 4, so its condition is at most 11 and a
# residual of 1e-10 ||b|| leaves x within 1.1e-9 of the solution; the other 1e-10 is the direct solve's and rounding's.
@pytest.mark.parametrize("shape", [(33, 65), (97, 129)])
def test_matrix_with_counts_to_seven(fg, ctx, shape):
    from scipy.sparse import diags
    from scipy.sparse.linalg import spsolve
    rng = np.random.default_rng(shape[0])
    I, J = shape
    on = np.zeros((I, J), bool)
    on[1:-1, 1:-1] = rng.random((I - 2, J - 2)) < 0.85
    nb = [np.roll(on, s, a) & on for s, a in ((1, 0), (-1, 0), (1, 1), (-1, 1))]   # i-1, i+1, j-1, j+1
    deg = sum(n.astype(int) for n in nb)
    count = np.where(on, deg + rng.integers(1, 4, on.shape), 0)
    assert count.max() == 7 and count.min() == 0
    code = np.where(on, 0x80 | (count << 4) | sum(n.astype(int) << k for k, n in enumerate(nb)), 0).astype(np.uint8)
    b = np.where(on, rng.standard_normal(on.shape), 0.0).ravel()
    A = diags([np.where(on, count, 1).ravel().astype(float), -(nb[1].ravel()[:-J].astype(float)),
               -(nb[0].ravel()[J:].astype(float)), -(nb[3].ravel()[:-1].astype(float)), -(nb[2].ravel()[1:].astype(float))],
              [0, J, -J, 1, -1], format="csc")
    x, st = np.zeros(I * J), fg.SolveStats()
    fg._check(fg.lib().fg_poisson_solve_matrix(ctx.h, I, J, code.ctypes.data, 1.0, b.ctypes.data, x.ctypes.data, 1e-10, 0,
                                               C.byref(st)))
    print(f"{shape}: {st.iterations} iterations", flush=True)
    assert st.converged and rel_l2(x, spsolve(A, b)) <= 1.2e-9
