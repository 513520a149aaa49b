"""Dataset kernels at the edges of their tiles and blocks: histograms equal the
oracle's exactly (whole counts), moments a float64 computation to the rounding
of their float result (one ulp, 2^-23 relative)."""

import numpy as np
import pytest

import oracle as O
from bayadera_amd import _lib, engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fac():
    f = engine.HipBayaderaFactory(0, 256)
    yield f
    f.release()


def _check(de, a):
    h, hr = de.histogram(a), O.histogram(a)
    assert np.array_equal(h.limits, hr.limits)
    assert np.array_equal(h.pdf, hr.pdf, equal_nan=True)
    assert np.array_equal(h.bin_ranks, hr.bin_ranks)
    x = a.astype(np.float64)
    assert np.allclose(de.data_mean(a), x.mean(0), rtol=2.0 ** -23, atol=np.abs(x).mean() * 1e-12)
    assert np.allclose(de.data_variance(a), x.var(0), rtol=2.0 ** -23, atol=0)


# one tile, a tile and a bit, one column per block, more columns than blocks,
# whole and partial rounds of eight loads; rows around the tiles of 1 to 64
@pytest.mark.parametrize("m,n", [(1, 511), (1, 513), (2, 256), (3, 129), (5, 4097), (8, 32768),
                                 (9, 65537), (33, 9000), (64, 4100), (65, 777), (4, 1048577)])
def test_estimates(fac, m, n):
    rng = np.random.default_rng([m, n])
    a = (rng.standard_normal((n, m)) * rng.uniform(0.1, 30.0, m) + rng.uniform(-50, 50, m)).astype(np.float32)
    _check(fac.dataset_engine(), a)


@pytest.mark.parametrize("scale", [1e-25, 1e-18, 1e18, 1e25])
def test_histogram_widths(fac, scale):
    """Rows narrower and wider than the width the bin's reciprocal takes."""
    a = (np.random.default_rng(4).standard_normal((5000, 3)) * np.float32(scale)).astype(np.float32)
    h, hr = fac.dataset_engine().histogram(a), O.histogram(a)
    assert np.array_equal(h.pdf, hr.pdf) and np.array_equal(h.bin_ranks, hr.bin_ranks)


def test_variance_with_far_first_values(fac):
    """A block's first value is its origin: far ones, and rows far from zero."""
    rng = np.random.default_rng(5)
    a = rng.standard_normal((300000, 2)).astype(np.float32)
    a[0, 0] = a[512 * 256, 0] = 3e4
    a[:, 1] += np.float32(1e5)
    _check(fac.dataset_engine(), a)


def test_non_finite_values(fac):
    a = np.random.default_rng(6).standard_normal((4000, 4)).astype(np.float32)
    a[17, 1], a[0, 2], a[3999, 3] = np.inf, np.nan, -np.inf
    de = fac.dataset_engine()
    with np.errstate(all="ignore"):
        x = a.astype(np.float64)
        assert np.array_equal(np.isnan(de.data_variance(a)), np.isnan(x.var(0)))
        mean = de.data_mean(a)
    assert np.isfinite(mean[0]) and mean[1] == np.inf and np.isnan(mean[2]) and mean[3] == -np.inf
    h, hr = de.histogram(a), O.histogram(a)
    assert np.array_equal(h.limits, hr.limits, equal_nan=True)
    assert np.array_equal(h.pdf, hr.pdf, equal_nan=True)


def test_leading_dimension(fac):
    """Rows of a wider matrix (ld > m) give what the rows alone give."""
    a = np.random.default_rng(7).standard_normal((3000, 7)).astype(np.float32)
    out = np.zeros(3, np.float32)
    _lib.call("bh_dataset_variance", fac.handle, a.ctypes.data, 3, 3000, 7, out.ctypes.data)
    assert np.array_equal(out, fac.dataset_engine().data_variance(np.ascontiguousarray(a[:, :3])))
    lim, pdf, rk = (np.zeros(s, np.float32) for s in ((3, 2), (3, 256), (3, 256)))
    _lib.call("bh_dataset_histogram", fac.handle, a.ctypes.data, 3, 3000, 7, lim.ctypes.data,
              pdf.ctypes.data, rk.ctypes.data)
    h = fac.dataset_engine().histogram(np.ascontiguousarray(a[:, :3]))
    assert np.array_equal(lim, h.limits) and np.array_equal(pdf, h.pdf) and np.array_equal(rk, h.bin_ranks)
