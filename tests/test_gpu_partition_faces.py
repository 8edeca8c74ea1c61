"""Face relaxation of the partitioned solve at the ends of its range: the
smallest blocks (3 nodes an axis: every face node is an edge node, and the
second neighbour of each lies outside), odd counts, and faces of 32761 nodes
(the largest a block may have is 32768), against the CPU oracle's form of the
same system: fields within 1e-9 s and the same passes, the bar of its
goldens."""
import numpy as np
import pytest

from fmm3d import lib, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [lib.ORDER_FIRST, lib.ORDER_MIXED])
@pytest.mark.parametrize("shape", [(6, 6, 6), (7, 6, 9), (17, 8, 66), (6, 361, 362)])
def test_partition_faces(shape, order):
    g = synth.make_grid(shape, 60.0, (2.0, 2.5), nv=(8, 8, 8))
    velv = synth.make_velv(g, 0.02, 4)
    face = synth.tele_bottom_face(g, synth.tele_sources(g, 2, 9)[1])
    ref, npass = O.relax_tele_part(g, velv, face, order)
    with lib.Context(g) as c:
        c.set_model(velv)
        c.solve_tele(face, order, lib.PREC_FP64, partition=True)
        d = float(np.abs(c.field(0) - ref).max())
        print(f"{shape} order {order}: {d:.2e} s, {npass} passes", flush=True)
        assert d <= 1e-9 and int(c.passes()[0]) == npass
