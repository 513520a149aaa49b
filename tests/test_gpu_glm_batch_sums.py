"""Accounted steps of a regression batch: the recorded means are the ensembles'
sums in the kernels' order, bit for bit, for dimensions around the groups of
four, 16 and 32 coordinates that a wave adds up together."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu


def _ensemble_mean(x):
    """x (W, d) float32: trees over 64 walkers, their sums pairwise in fours, those in turn."""
    s = x.reshape(-1, 64, x.shape[1])
    for i in (32, 16, 8, 4, 2, 1):
        s = s[:, :i] + s[:, i:2 * i]
    w = s[:, 0].reshape(-1, 4, x.shape[1])
    total = np.zeros(x.shape[1], np.float32)
    for b in (w[:, 0] + w[:, 1]) + (w[:, 2] + w[:, 3]):
        total = total + b
    return total / np.float32(x.shape[0])


@pytest.mark.parametrize("prec", [_lib.BH_GLM_FP16X2, _lib.BH_GLM_FP32])
@pytest.mark.parametrize("walkers", [512, 2048])
def test_recorded_means(walkers, prec):
    rng = np.random.default_rng(walkers)
    dims = [1, 3, 4, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64]
    codes = [rng.integers(0, 100, (50 + d, d)).astype(np.uint8) for d in dims]
    scales = [(rng.uniform(0.5, 2.0, d) / 448).astype(np.float32) for d in dims]
    labels = [(rng.random(50 + d) < 0.5).astype(np.float32) for d in dims]
    fac = engine.HipBayaderaFactory(0, 256)
    bt = fac.glm_batch(models.GlmBatchModel(codes, scales, labels, 5.0), walkers).set_precision(prec)
    lim = np.zeros((len(dims), 64, 2), np.float32)
    lim[:, :, 0], lim[:, :, 1] = -1.0, 2.0
    bt.init_position(5, lim)
    before = bt.state()[0]
    series = np.empty(sum(dims), np.float32)
    bt.run(6, 1, 2.0, series=series)
    xs = bt.state()[0]
    at = 0
    for p, d in enumerate(dims):
        assert not np.array_equal(before[p], xs[p])
        assert np.array_equal(series[at:at + d], _ensemble_mean(np.asarray(xs[p], np.float32).reshape(walkers, -1)[:, :d])), d
        at += d
    bt.release()
    fac.release()
