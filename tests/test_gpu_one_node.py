"""8 x 8 patches walked one node per lane and by the walk of the other patch
shapes (which layers too large for 32-bit offsets take): the same passes in
the same order, so the same fields.  Float64 to the bit (one fixed point per
node); float32 to the bit where every sweep is ordered (plane waves), and
within its bar of 1 ms for local sources, whose sweeps are not.  Patches with
remainders 1 and 7, batches below and above the eight placed by XCD, replayed
and direct sweeps, refined blocks."""
import numpy as np
import pytest

from fmm3d import lib, synth

pytestmark = pytest.mark.gpu


def _both(c, solve, nsrc):
    out = []
    for one in (1, 0):
        c.set_option("one_node", one)
        solve()
        out.append([c.field(q) for q in range(nsrc)])
    return out


@pytest.mark.parametrize("graph", [1, 0])
@pytest.mark.parametrize("nsrc", [3, 9])
def test_plane_waves(nsrc, graph):
    g = synth.make_grid((14, 33, 39), 90.0, (3.0, 3.5), nv=(8, 8, 8))
    faces = np.stack([synth.tele_bottom_face(g, s) for s in synth.tele_sources(g, nsrc, 7)])
    with lib.Context(g) as c:
        c.set_model(synth.make_velv(g, 0.03, 7))
        c.set_option("graph", graph)
        for prec in (lib.PREC_FP64, lib.PREC_FP32):
            for order in (lib.ORDER_MIXED, lib.ORDER_FIRST):
                a, b = _both(c, lambda: c.solve_tele(faces, order, prec), nsrc)
                for q in range(nsrc):
                    assert np.array_equal(a[q], b[q]), (prec, order, q)


def test_local_sources():
    g = synth.make_grid((25, 33, 39), 120.0, (3.0, 3.5), nv=(8, 8, 8))
    src = np.stack([synth.point_source_rad(g, s) for s in synth.local_sources(g, 2, 5, radius_range=(5, 5))])
    with lib.Context(g) as c:
        c.set_model(synth.make_velv(g, 0.03, 5))
        for prec, tol in ((lib.PREC_FP64, 1e-9), (lib.PREC_FP32, 1e-3)):
            a, b = _both(c, lambda: c.solve_point(src, 5, 5, precision=prec), 2)
            d = max(float(np.abs(a[q] - b[q]).max()) for q in range(2))
            print(f"precision {prec}: {d:.2e} s", flush=True)
            assert d <= tol


def test_one_node_range():
    g = synth.make_grid((5, 9, 9), 60.0, (2.0, 2.5), nv=(8, 8, 8))
    with lib.Context(g) as c:
        for bad in (-1, 2):
            with pytest.raises(lib.FmmError):
                c.set_option("one_node", bad)
