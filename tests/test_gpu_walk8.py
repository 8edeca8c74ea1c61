"""The 8 x 8 column walk's placement of slots: in a first sweep a multiple of
eight of them run on one XCD each and the rest are spread, so a batch's
fields must not depend on how many there are or on a slot's place among them.
Each source of a batch equals the same source solved alone: float64 exactly
(the walk's fixed point has one value per node, whatever the order), float32
too (every first sweep is ordered, and the passes are the same).  Patches
with remainders 1 and 7; the serving loop, whose slots join in any sweep,
within the float32 bound of 1 ms."""
import numpy as np
import pytest

from fmm3d import lib, synth

pytestmark = pytest.mark.gpu


def _case(nsrc):
    g = synth.make_grid((14, 33, 39), 90.0, (3.0, 3.5), nv=(8, 8, 8))
    velv = synth.make_velv(g, 0.03, 7)
    faces = np.stack([synth.tele_bottom_face(g, s) for s in synth.tele_sources(g, nsrc, 7)])
    return g, velv, faces


@pytest.mark.parametrize("precision", [lib.PREC_FP64, lib.PREC_FP32])
@pytest.mark.parametrize("nsrc", [7, 8, 11, 17])
def test_batch_fields_equal_the_sources_alone(nsrc, precision):
    g, velv, faces = _case(17)
    with lib.Context(g) as c:
        c.set_model(velv)
        c.solve_tele(faces[:nsrc], lib.ORDER_MIXED, precision)
        batch = [c.field(q) for q in range(nsrc)]
        for q in (0, nsrc // 2, nsrc - 1):
            c.solve_tele(faces[q], lib.ORDER_MIXED, precision)
            assert np.array_equal(c.field(0), batch[q]), (nsrc, q)


def test_served_batches_of_eight_and_more():
    g, velv, faces = _case(13)
    rcv = synth.receivers_rad(synth.receivers(g, 12, 7))
    with lib.Server(hbm_budget=4e9, max_slots=16) as srv:
        tickets = [srv.submit(g, velv, 1, faces=faces[a:b], rcv=rcv) for a, b in ((0, 4), (4, 9), (9, 13))]
        times = []
        for t in tickets:
            assert srv.wait(t, 60.0)
            times.append(srv.result(t)[0])
    with lib.Context(g) as c:
        c.set_model(velv)
        c.solve_tele(faces, lib.ORDER_MIXED, lib.PREC_FP32)
        assert np.abs(np.concatenate(times).astype(np.float64) - c.receivers(rcv)).max() <= 1e-3
