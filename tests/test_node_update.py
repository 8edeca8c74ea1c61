"""The walks' node update on the CPU: the update that takes one octant where
that one is certain, and each lane's own octants where it is not, gives the
bits of the minimum over all eight in the same arithmetic.  Random stencils of
waves with noise and kinks: ties (values on a coarse grain, equal neighbours),
both sides of an axis counted, clamped discriminants, sides outside the grid,
unknown neighbours and centres.  In float32 with exact and with hardware-like
square roots and reciprocals (a unit in the last place off, by the argument),
and both forms: one octant first, and all eight at once."""
import ctypes

import pytest

import native_lib

N = 400_000


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return native_lib.load("node_update", tmp_path_factory.mktemp("native"))


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("f32,ulp", [(0, 0), (1, 0), (1, 1), (1, 7)])
def test_update_is_the_least_of_eight_octants(so, f32, ulp, order):
    out = (ctypes.c_longlong * 6)()
    so.node_update.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_uint, ctypes.c_int,
                               ctypes.POINTER(ctypes.c_longlong)]
    so.node_update(f32, order, N, 11 + 2 * ulp + order, ulp, out)
    differ, two, clamped, ties, unknown, outside = out
    print(f"float{32 if f32 else 64} order {order}: {differ} differ; {two} two-sided, {clamped} clamped, {ties} ties, "
          f"{unknown} unknown, {outside} with a side outside")
    # every kind of node is among them
    assert min(two, ties, unknown, outside) > N // 100 and (not f32 or clamped > N // 100)
    assert differ == 0
