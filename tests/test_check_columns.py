"""The fixed-point check's look, on the CPU: no wavefront of it reads a column
outside its slot.  A slot gets whole blocks of 256 columns, so where its
columns modulo 256 are 1 to 192 its last block has wavefronts without any,
and a read of theirs in the last layer of the last slot would lie beyond the
fields' allocation.  Every lane's column (its own, and each late input) is
formed with the kernel's functions; the column is the same in both precisions
and every layer."""
import ctypes
import itertools

import pytest

import native_lib


@pytest.fixture(scope="module")
def extent(tmp_path_factory):
    so = native_lib.load("look_columns", tmp_path_factory.mktemp("native"))

    def call(*args):
        out = (ctypes.c_longlong * 4)()
        so.look_extent(*args, out)
        return list(out)
    call.fits = so.look_fits
    return call


# columns modulo 256: 0, 1, 64, 129, 192, 193, 255 and small slots
SHAPES = [(16, 16), (32, 24), (19, 27), (25, 13), (200, 200), (129, 129), (65, 65), (110, 140), (201, 201), (321, 321),
          (16, 28), (193, 1), (64, 7), (51, 5), (3, 3), (3, 300), (300, 3)]


def test_shapes_cover_the_remainders():
    assert {0, 1, 64, 129, 192, 193, 255} <= {x * z % 256 for x, z in SHAPES}


@pytest.mark.parametrize("nnx,nnz", SHAPES)
def test_every_column_read_is_the_slots(extent, nnx, nnz):
    for px, pz in ((8, 8), (8, 16), (16, 8), (64, 8), (32, 32)):
        for fx, fz in itertools.product((-1, 0, 1), repeat=2):
            for snx, snz in ((nnx, nnz), (max(1, nnx - 1), nnz), (nnx, max(1, nnz - 9)), (max(1, nnx // 2), max(1, nnz // 3))):
                lo, hi, own, wrong = extent(nnx, nnz, snx, snz, px, pz, fx, fz)
                assert lo >= 0 and hi < nnx * nnz, (px, pz, fx, fz, snx, snz, lo, hi)
                assert own == snx * snz and wrong == 0


@pytest.mark.parametrize("nbytes", [4, 8])
def test_offsets_of_long_rows_fit(extent, nbytes):
    """An offset in 32 bits of bytes is the exact one whatever the rows' length."""
    edge = ((1 << 32) - 1) // nbytes // 4 - 16   # the longest rows counted from two rows before
    for nnz in (3, 140, 65536, edge - 1, edge, edge + 1, 1 << 27, 1 << 28, (1 << 29) + 5, (1 << 31) - 1):
        assert extent.fits(nnz, nbytes), nnz
