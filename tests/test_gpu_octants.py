"""Node updates decided by one octant, or by all eight where that one is not
certain: boundary times that put many nodes on the line between the two --
a flat face (no lateral slope at all: ties), slopes along one axis only, a
ridge and a trough (both sides of an axis count) and a steep tilt -- against
the CPU oracle's single-phase relaxation, which always takes the minimum
over eight.  Float64 relaxes to the same values up to the sweeps' own settle
tolerance (1e-14 of times near 500 s, over some hundred dependent nodes:
1e-9 s); float32 within 1 ms, the bound of that path."""
import numpy as np
import pytest

from fmm3d import lib, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _face(kind, nx, nz):
    x, z = np.meshgrid(np.arange(nx) - nx // 2, np.arange(nz) - nz // 2, indexing="ij")
    return 500.0 + {"flat": 0.0 * x, "theta": 0.4 * x + 0.0 * z, "phi": -0.3 * z + 0.0 * x,
                    "ridge": -0.35 * np.abs(x) + 0.1 * z, "trough": 0.35 * np.abs(x) + 0.2 * np.abs(z),
                    "tilt": 0.5 * x + 0.45 * z}[kind]


@pytest.mark.parametrize("order", [lib.ORDER_FIRST, lib.ORDER_MIXED])
@pytest.mark.parametrize("kind", ["flat", "theta", "phi", "ridge", "trough", "tilt"])
def test_one_octant_gives_the_eight_octants_field(kind, order):
    # patches of 8 with remainders 1 and 7
    g = synth.make_grid((12, 25, 31), 60.0, (2.0, 2.5), nv=(8, 8, 8))
    velv = synth.make_velv(g, 0.02, 3)
    face = _face(kind, g.nnx, g.nnz)
    ref, _ = O.relax1_tele(g, O.gridder(g, velv), face, order)
    with lib.Context(g) as c:
        c.set_model(velv)
        for prec, tol in ((lib.PREC_FP64, 1e-9), (lib.PREC_FP32, 1e-3)):
            c.solve_tele(face, order, prec)
            d = float(np.abs(c.field(0) - ref).max())
            print(f"{kind} order {order} precision {prec}: {d:.2e} s", flush=True)
            assert d <= tol
