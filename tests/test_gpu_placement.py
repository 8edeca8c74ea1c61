"""First sweeps of eight sources, whose patches are meant to run on one XCD
per source and pass values on through its L2, where they do not: patches of a
source spread over the XCDs on purpose.  A patch then reads its neighbours
late, in no order, or not before its bounded wait ends; the source counts as
out of order, the check looks at every neighbour, and further sweeps settle
the same fixed point.  Against the CPU oracle's relaxation: float64 within
1e-9 s (sweeps settle to 1e-14 of times near 500 s over some hundred dependent
nodes), float32 within its bar of 1 ms.  Faces whose waves run along the
patches' order either way, and meet in a trough; all settle in the oracle's
node-by-node relaxation, that is, have one fixed point (a ridge that is tilted
as well has none, and its field depends on the order anywhere)."""
import numpy as np
import pytest

from fmm3d import lib, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("skew", [1, 3, 4])
def test_a_placement_that_does_not_hold_changes_no_result(skew):
    g = synth.make_grid((12, 33, 39), 60.0, (2.0, 2.5), nv=(8, 8, 8))
    velv = synth.make_velv(g, 0.08, 7)
    x, z = np.meshgrid(np.arange(g.nnx) - g.nnx // 2, np.arange(g.nnz) - g.nnz // 2, indexing="ij")
    faces = np.stack([500.0 + v * 0.3 * np.abs(x) + a * x + b * z for v, a, b in
                      ((-1, 0.0, 0.1), (0, 0.0, 0.1), (0, 0.2, 0.2), (0, -0.25, 0.05), (0, -0.1, -0.2), (1, 0.0, 0.1),
                       (1, 0.2, 0.2), (1, -0.25, 0.05))])
    veln = O.gridder(g, velv)
    ref = [O.relax1_tele(g, veln, f, lib.ORDER_MIXED)[0] for f in faces]
    with lib.Context(g) as c:
        c.set_model(velv)
        c.set_option("spin_limit", 500)   # a wait across XCDs ends soon
        c.set_option("placement_skew", skew)
        for prec, tol in ((lib.PREC_FP64, 1e-9), (lib.PREC_FP32, 1e-3)):
            c.solve_tele(faces, lib.ORDER_MIXED, prec)
            d = max(float(np.abs(c.field(s) - ref[s]).max()) for s in range(8))
            print(f"skew {skew} precision {prec}: {d:.2e} s, {c.stats()['sweeps']} sweeps", flush=True)
            assert d <= tol


def test_placement_skew_range():
    g = synth.make_grid((5, 9, 9), 60.0, (2.0, 2.5), nv=(8, 8, 8))
    with lib.Context(g) as c:
        for bad in (-1, 8):
            with pytest.raises(lib.FmmError):
                c.set_option("placement_skew", bad)
