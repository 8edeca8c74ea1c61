"""The LDS cells of an 8 x 8 patch, on the CPU: lanes without a node (patches
with a remainder) read a stencil of spare cells, all of them in the array; no
two lanes write one cell of the patch or its halo; a node's stencil is its
neighbours' cells.  Every remainder, patches at each edge of the grid and
inside it."""
import ctypes
import itertools

import pytest

import native_lib


@pytest.fixture(scope="module")
def cells(tmp_path_factory):
    so = native_lib.load("patch8_cells", tmp_path_factory.mktemp("native"))

    def call(*args):
        out = (ctypes.c_int * 4)()
        so.patch8_cells(*args, out)
        return list(out)
    return call


@pytest.mark.parametrize("nx", range(1, 9))
def test_every_cell_is_in_the_array(cells, nx):
    for nz in range(1, 9):
        # rows and columns of the grid before the patch, and behind a whole one
        for before_x, before_z in itertools.product((0, 2), repeat=2):
            for behind_x, behind_z in itertools.product((0, 1, 2) if nx == 8 else (0,), (0, 1, 2) if nz == 8 else (0,)):
                lo, hi, size, faults = cells(nx, nz, -before_x, nx - 1 + behind_x, -before_z, nz - 1 + behind_z)
                assert lo >= 0 and hi < size, (nx, nz, lo, hi, size)
                assert faults == 0
