"""Matrix products over lists that are short on average (a lane each, up to 32
entries, the longer ones sixteen lanes each): lengths around 32 and around the
64 entries sixteen lanes take at a time, one to nine long lists among a
wavefront's 64, counts of lists that are no multiple of 64 or 256, empty
lists, infinities and NaN among the values; also just below and at the mean
length where the kernels change.  Against the oracle's float32 sums in
subinv's order: bit for bit."""
import numpy as np
import pytest

from fmm3d import lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(lens, ncols, seed, special):
    rng = np.random.default_rng(seed)
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


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("nlists", [63, 256, 1001])
def test_short_rows(nlists, special):
    rng = np.random.default_rng(nlists)
    lens = rng.integers(0, 4, nlists)
    # longer ones: one in the first wavefront, nine in the last
    lens[5] = 33
    lens[-9:] = [31, 32, 33, 63, 64, 65, 129, 0, 40] if nlists > 100 else [31, 32, 33, 34, 0, 1, 35, 36, 33]
    assert lens.sum() < 8 * nlists
    _check(list(lens), 500, nlists, special)


def test_short_columns():
    # few rows over many columns: most columns empty; one row holds every column, two hold half
    rng = np.random.default_rng(9)
    _check([3000, 1500, 1500] + list(rng.integers(0, 300, 20)), 3000, 9, False)


@pytest.mark.parametrize("last", [7, 8])
def test_either_side_of_the_rule(last):
    # 300 rows of 8 entries but the last: below 8 on average, or 8
    _check([8] * 299 + [last], 200, last, False)
