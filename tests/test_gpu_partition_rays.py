"""Rays of a partitioned solve end at the grid's faces, whatever the context
solved before: after a solve of point sources, whose rays end at the source,
the partitioned solve's rows are those of a new context, entry for entry."""
import numpy as np
import pytest

import goldens as G
from fmm3d import lib

pytestmark = pytest.mark.gpu


def test_partitioned_rays_after_point_sources():
    gd = G.load("tele_31x33x35_mixed")
    g = gd.g
    src = np.array([[-0.4 * (g.nnr - 1) * g.dnr, g.rgox + 0.45 * (g.nnx - 1) * g.dnx, g.rgoz + 0.55 * (g.nnz - 1) * g.dnz]] * 2)
    rows = []
    for point_first in (False, True):
        with lib.Context(g) as c:
            c.set_model(gd.velv)
            if point_first:
                c.solve_point(src, 2, 2, lib.ORDER_MIXED, lib.PREC_FP64)
            c.solve_tele(gd.faces[:2], gd.fom, lib.PREC_FP64, partition=True)
            rows.append(c.frechet(gd.rcv))
    for a, b in zip(*rows):
        assert np.array_equal(a, b)
