"""acor split over the chip: every level, slice and tree against the oracle's
one-slice-at-a-time estimator, bit for bit (the sums keep its shape, so there
is no tolerance)."""
import numpy as np
import pytest

import oracle as O
from bayadera_amd import engine

pytestmark = pytest.mark.gpu


def _walk(n, dim, seed):
    """Columns from white noise to a random walk: the estimator stops at the
    first level, at a deep one and at the last."""
    rng = np.random.default_rng([seed, n, dim])
    e = rng.standard_normal((n, dim))
    w = np.cumsum(e, axis=0)
    mix = np.linspace(0.0, 1.0, dim) if dim > 1 else np.ones(1)
    return ((1.0 - mix) * e + mix * w + 3.0).astype(np.float32)


def _equal(got, want):
    assert np.array_equal(got.tau, want.tau, equal_nan=True)
    assert np.array_equal(got.mean, want.mean, equal_nan=True)
    assert np.array_equal(got.sigma, want.sigma, equal_nan=True)


# around the line of the rule, the slice (256), the pyramid's blocks (2048 and
# 2048 x 2048 / 2), odd lengths at several levels; dimensions around the mean's
# group rule (16) and its odd groups (3, 7)
@pytest.mark.parametrize("n,dim", [(160, 2), (161, 5), (257, 1), (511, 3), (513, 7), (2047, 16), (2048, 17),
                                   (2049, 2), (4097, 5), (22529, 3), (65535, 2), (104448, 1),
                                   (106497, 2)])
def test_acor_split_equals_oracle(n, dim):
    fac = engine.HipBayaderaFactory(0, 256)
    x = _walk(n, dim, 1)
    _equal(fac.acor_engine().acor(x), O.acor(x))
    fac.release()


@pytest.mark.parametrize("wgs", [64, 128, 512, 1024])
def test_acor_split_work_groups(wgs):
    fac = engine.HipBayaderaFactory(0, wgs)
    for n, dim in ((1025, 1), (3071, 18), (9999, 4)):
        x = _walk(n, dim, 2)
        _equal(fac.acor_engine().acor(x), O.acor(x, wgs))
    fac.release()


def test_acor_split_leaves_the_series_alone_and_takes_non_finite_values():
    import torch
    fac = engine.HipBayaderaFactory(0, 256)
    x = _walk(3000, 3, 3)
    x[5, 0] = np.inf
    x[7, 1] = np.nan
    d = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    _equal(fac.acor_engine().acor(d), O.acor(x))
    assert np.array_equal(d.cpu().numpy(), x, equal_nan=True)
    fac.release()


def test_acor_split_batch_equals_each_series():
    fac = engine.HipBayaderaFactory(0, 256)
    dims, n = [1, 2, 5, 16, 23], 1500
    xs = [_walk(n, d, 4 + d) for d in dims]
    got = fac.acor_engine().acor_batch(np.concatenate([x.reshape(-1) for x in xs]), dims, n)
    for x, g in zip(xs, got):
        _equal(g, O.acor(x))
    fac.release()
