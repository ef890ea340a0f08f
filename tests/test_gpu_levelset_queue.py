"""The level set and the velocity extrapolation where their queues and lists are full: many blobs of liquid, so that more
tiles are queued for a band than a launch has blocks and a region row holds many cells of one level, against the oracle."""
import ctypes as C

import numpy as np
import pytest
from helpers import assert_substep_parity, oracle_state_dict

pytestmark = pytest.mark.gpu


def _blobs(orc, fg, I, J, period, size, ppc=2, seed=3):
    """A scene of solid-free blobs of size x size cells every `period` cells, two particles a cell, inside walls."""
    dx = 1.0 / max(I, J)
    p = orc.make_params(I, J, dx=dx, ppc=ppc, tol=1e-12)
    walls = [fg.box(0, dx, 0, J * dx), fg.box((I - 1) * dx, I * dx, 0, J * dx), fg.box(0, I * dx, 0, dx),
             fg.box(0, I * dx, (J - 1) * dx, J * dx)]
    fluids = [fg.box(i * dx, (i + size) * dx, j * dx, (j + size) * dx)
              for i in range(2, I - size - 1, period) for j in range(2, J - size - 1, period)]
    return p, orc.init_scene(p, walls, fluids, seed=seed)


# 21 x 20 tiles whose blobs all reach the band's last level (>= 16 cells deep): a queue of over 256 tiles; the same with
# ragged sides; blobs of 2 cells every 4 (rows of 16 cells of one level)
@pytest.mark.parametrize("I,J,period,size", [(641, 660, 42, 38), (161, 97, 4, 2), (33, 65, 7, 3)])
def test_many_blobs(orc, fg, ctx, I, J, period, size):
    p, st = _blobs(orc, fg, I, J, period, size)
    dt = np.float32(1.0 / 60)
    with fg.Scene(ctx, fg.make_params(I, J, dx=1.0 / max(I, J), ppc=2, tol=1e-10, max_particles=I * J * 4)) as sc:
        sc.set_friction(np.zeros(4, np.float32))
        sc.set_state(oracle_state_dict(st))
        sc.substep(float(dt))
        g = sc.get_state()
    orc.lib().orc_substep(C.byref(p), st.ref(), C.c_float(dt), C.byref(orc.OrcStats()))
    assert_substep_parity(g, st, print, what=f"{I}x{J}/{period}")
