"""The check after the first sweep (which nodes would still move) over layer
counts around its four layers at a time and lateral sizes around a wavefront,
a block and a patch: waves that cross the patches' order both ways (a ridge, a
trough and a near-vertical wave in a rough model), two slots that end at
different sweeps.  A node it misses would leave the field short of the oracle's
fixed point: float64 within 1e-9 s (sweeps settle to 1e-14 of times near 500 s
over some hundred dependent nodes), float32 within its bar of 1 ms."""
import numpy as np
import pytest

from fmm3d import lib, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 17, 15), (4, 16, 16), (5, 8, 33), (6, 65, 4), (7, 9, 57), (13, 31, 25)])
def test_check_finds_what_moves(shape):
    g = synth.make_grid(shape, 60.0, (2.0, 2.5), nv=(8, 8, 8))
    velv = synth.make_velv(g, 0.08, 7)
    x, z = np.meshgrid(np.arange(g.nnx) - g.nnx // 2, np.arange(g.nnz) - g.nnz // 2, indexing="ij")
    faces = np.stack([500.0 - 0.3 * np.abs(x) + 0.1 * z, 500.0 + 0.3 * np.abs(x) + 0.25 * np.abs(z), 500.0 + 0.02 * x - 0.01 * z,
                      500.0 + 0.3 * x + 0.2 * z])
    veln = O.gridder(g, velv)
    ref = [O.relax1_tele(g, veln, f, lib.ORDER_MIXED)[0] for f in faces]
    with lib.Context(g) as c:
        c.set_model(velv)
        for prec, tol in ((lib.PREC_FP64, 1e-9), (lib.PREC_FP32, 1e-3)):
            c.solve_tele(faces, lib.ORDER_MIXED, prec)
            for s in range(len(faces)):
                d = float(np.abs(c.field(s) - ref[s]).max())
                print(f"{shape} precision {prec} face {s}: {d:.2e} s", flush=True)
                assert d <= tol
