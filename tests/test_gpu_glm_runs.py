"""Logistic log posteriors with short runs of rows shared between the
work-groups of a round, and with one run each."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu


# fewer rows than a round's work-groups, runs that do and do not divide among
# them, a last run of one row, runs too long to be shared
@pytest.mark.parametrize("N,d,n", [(1, 32, 5), (700, 64, 256), (50021, 32, 1024), (50049, 64, 300),
                                   (65537, 32, 4096), (400001, 32, 512)])
def test_short_runs(N, d, n):
    """Per row: the split coefficients carry 21 bits (fp16 x 2; 24 for bf16 x 3),
    the float sums of a row's d products and of its run's terms d + 24
    roundings of the terms' size."""
    rng = np.random.default_rng([N, d, n])
    X = models.to_bf16(rng.standard_normal((N, d)).astype(np.float32) / np.sqrt(d)).reshape(N, d)
    y = (rng.random(N) < 0.5).astype(np.float32)
    pts = rng.standard_normal((n, d)).astype(np.float32)
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.glm_logistic_model(X, y, 5.0))
    ref = sf.log_density(pts, _lib.BH_GLM_FP64)
    x64 = np.abs(models.from_bf16(X).reshape(N, d).astype(np.float64))
    size = np.abs(pts.astype(np.float64)) @ x64.sum(0) + N
    tol = ((d + 24) * 2.0 ** -24 + 2.0 ** -21) * size
    for prec in (_lib.BH_GLM_FP16X2, _lib.BH_GLM_BF16X3):
        assert np.all(np.abs(sf.log_density(pts, prec) - ref) <= tol), prec
    sf.release()
    fac.release()
