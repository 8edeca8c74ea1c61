"""Batches of more sources than the listing of a sweep's slots takes at a time
(256 threads up to 256 slots, 1024 beyond): every slot of a batch holds the
field of its source solved alone.  Float64 exactly (one fixed point per
node), float32 too (every first sweep is ordered).  Sources that end at
different sweeps, on layers above and below the 64 nodes from which a slot is
placed on one XCD, with and without captured sweeps."""
import numpy as np
import pytest

from fmm3d import lib, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [1, 0])
@pytest.mark.parametrize("nsrc", [256, 257, 1030])
@pytest.mark.parametrize("shape", [(6, 9, 11), (5, 7, 9)])
def test_every_slot_is_its_source_alone(shape, nsrc, graph):
    g = synth.make_grid(shape, 60.0, (1.0, 1.2), nv=(8, 8, 8))
    x, z = np.meshgrid(np.arange(g.nnx) - g.nnx // 2, np.arange(g.nnz) - g.nnz // 2, indexing="ij")
    kinds = np.stack([500.0 + v * np.abs(x) + a * x + b * z for v, a, b in
                      ((0.0, 0.3, 0.1), (0.0, -0.2, 0.25), (0.3, 0.0, 0.1), (-0.3, 0.0, 0.1), (0.0, 0.0, 0.0))])
    of = np.arange(nsrc) % len(kinds)
    with lib.Context(g) as c:
        c.set_model(synth.make_velv(g, 0.05, 7))
        c.set_option("graph", graph)
        for prec in (lib.PREC_FP64, lib.PREC_FP32):
            alone = []
            for f in kinds:
                c.solve_tele(f, lib.ORDER_MIXED, prec)
                alone.append(c.field(0))
            c.solve_tele(kinds[of], lib.ORDER_MIXED, prec)
            for q in [0, 1, 2, 3, 4, 63, 64, 255, nsrc - 2, nsrc - 1] + list(range(5, nsrc, 37)):
                assert np.array_equal(c.field(q), alone[of[q]]), (prec, q)
