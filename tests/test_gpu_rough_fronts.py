"""Nodes where the full octant is not the least: boundary times that jump by
about a cell's traveltime between neighbours leave sides that enter late or
with the wrong sign, discriminants below zero, both sides of an axis and ties.

The solves take the minimum over a node's octants there, and must leave what
the CPU oracle's full enumeration leaves: the partitioned march (its value per
node depends on the neighbours only) within 1e-9 s with the same passes, the
bar of its goldens; the one-domain float64 relaxation within the same bar, in
first order (in mixed order such fronts have no one-domain fixed point)."""
import numpy as np
import pytest

from fmm3d import lib, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(kind, shape):
    g = synth.make_grid(shape, 60.0, (2.0, 2.5), nv=(8, 8, 8))
    rng = np.random.default_rng(11)
    x, z = np.meshgrid(np.arange(g.nnx), np.arange(g.nnz), indexing="ij")
    face = 500.0 + 0.3 * x + 0.2 * z
    if kind == "steps":
        face = face + 0.5 * ((x // 2 + z // 3) % 2)
    elif kind == "noise":
        face = face + rng.uniform(0.0, 0.5, face.shape)
    else:   # spikes: single early nodes
        face = face - 0.5 * (rng.uniform(size=face.shape) < 0.06)
    return g, synth.make_velv(g, 0.1, 5), face


@pytest.mark.parametrize("order", [lib.ORDER_FIRST, lib.ORDER_MIXED])
@pytest.mark.parametrize("kind", ["steps", "noise", "spikes"])
@pytest.mark.parametrize("shape", [(9, 18, 17), (13, 27, 34)])
def test_rough_fronts(kind, order, shape):
    g, velv, face = _case(kind, shape)
    part, npass = O.relax_tele_part(g, velv, face, order)
    with lib.Context(g) as c:
        c.set_model(velv)
        c.solve_tele(face, order, lib.PREC_FP64, partition=True)
        d = float(np.abs(c.field(0) - part).max())
        print(f"{kind} order {order} {shape}: partitioned {d:.2e} s, {npass} passes", flush=True)
        assert d <= 1e-9 and int(c.passes()[0]) == npass
        if order == lib.ORDER_FIRST:
            ref, _ = O.relax1_tele(g, O.gridder(g, velv), face, order)
            c.solve_tele(face, order, lib.PREC_FP64)
            d = float(np.abs(c.field(0) - ref).max())
            print(f"    one domain {d:.2e} s", flush=True)
            assert d <= 1e-9
