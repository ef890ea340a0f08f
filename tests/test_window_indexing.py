"""Index arithmetic of the level-0 tiles of k_mg_up0 and k_pcg_dir: the header that the kernels use (fg_tiles.h), compiled
for the host and replayed over many grids and tilings.  Every cell is one tile's, every tile one block's, a staged position
holds the cell that the stencil or the matrix row reads there, and the level-1 patch holds the parents that the
interpolation takes."""
import ctypes as C
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tiles") / "libtiles.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall",
                    "-I", os.path.join(HERE, "..", "flipsolver2d_amd", "csrc"), os.path.join(HERE, "tile_index_check.cpp"),
                    "-o", out], check=True)
    return C.CDLL(out).check_tiles


def _cases():
    fixed = [(64, 64, 1024, 1024), (100, 37, 1024, 1024), (5, 3, 256, 4096), (257, 300, 4096, 7), (64, 4096, 2048, 1024),
             (2, 2, 1024, 1), (31, 33, 256, 2), (32, 32, 1024, 1), (33, 32, 1024, 1), (1024, 40, 512, 4096), (4, 3000, 1024, 5)]
    rng = random.Random(3)
    for _ in range(25):
        fixed.append((rng.randint(2, 260), rng.randint(2, 400), rng.choice([256, 1024, 4096]), rng.randint(1, 200)))
    return fixed


@pytest.mark.parametrize("I,J,min_chunk,most", _cases())
def test_tiles_own_and_stage_their_cells(check, I, J, min_chunk, most):
    assert check(I, J, min_chunk, most) == 0
