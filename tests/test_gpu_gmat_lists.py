"""Matrix products over rows and columns whose lengths end before, at and after
the 64 entries a wavefront takes at a time (none, 1, 63, 64, 65, 127, 128, 129,
one that holds every column), with infinities and NaN among the values, against
the oracle's float32 sums in subinv's order: bit for bit."""
import numpy as np
import pytest

from fmm3d import lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("special", [False, True])
def test_list_lengths(special):
    rng = np.random.default_rng(3)
    ncols = 1000
    lens = [0, 1, 63, 64, 65, 0, 127, 128, 129, 1000, 7, 8, 9] + list(rng.integers(0, 200, 400))
    cols = np.concatenate([np.sort(rng.choice(ncols, n, replace=False)) + 1 for n in lens]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    vals = (rng.normal(size=len(cols)) * 10.0 ** rng.integers(-6, 6, len(cols))).astype(np.float32)
    if special:
        vals[rng.integers(0, len(vals), 12)] = [np.inf, -np.inf, np.nan, -0.0] * 3
    d = rng.normal(size=len(lens)).astype(np.float32)
    a = rng.normal(size=ncols).astype(np.float32)
    cd = rng.uniform(0.5, 2.0, size=len(lens)).astype(np.float32)
    with lib.FrechetMatrix(rp, cols, vals, ncols) as m:
        for got, ref in ((m.gtx(d), O.gmat_gtx(rp, cols, vals, ncols, d)), (m.gx(a, cd), O.gmat_gx(rp, cols, vals, a, cd)),
                         (m.gx(a), O.gmat_gx(rp, cols, vals, a))):
            assert np.array_equal(got, ref, equal_nan=True)
            assert np.array_equal(np.signbit(got[~np.isnan(got)]), np.signbit(ref[~np.isnan(ref)]))
