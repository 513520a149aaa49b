"""Edges of the likelihood kernels' tiles: rows around the 16-row blocks,
features around the padded 16, 32 and 64, points that do and do not fill a
launch."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("d", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,n", [(1, 1), (15, 256), (16, 257), (17, 40), (513, 300), (4097, 1000)])
def test_linear_regression_tiles(N, n, d):
    """The fp32 residual of a row is y - t with t a chain of d products, each
    rounding once: |error| <= (d + 1) eps (sum |x b| + |y|); its square and
    the sum of four add 5 eps of the square.  The rest is in double."""
    rng = np.random.default_rng([N, n, d])
    X = rng.standard_normal((N, d)).astype(np.float32)
    beta = rng.standard_normal(d)
    y = (X @ beta + 0.3 * rng.standard_normal(N)).astype(np.float32)
    pts = np.concatenate([beta + 0.1 * rng.standard_normal((n, d)), 0.2 * rng.standard_normal((n, 1)) - 1.0],
                         1).astype(np.float32)
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.glm_gaussian_model(X, y, 10.0, 1.0))
    x64, y64 = X.astype(np.float64), y.astype(np.float64)
    b, ls = pts[:, :d].astype(np.float64), pts[:, d].astype(np.float64)
    r = y64[None, :] - b @ x64.T
    w = 0.5 * np.exp(-2 * ls)
    ref = (-N * (ls + 0.5 * np.log(2 * np.pi)) - w * np.sum(r * r, 1)
           - 0.5 * (np.sum(b * b, 1) / 100.0 + ls ** 2))
    e = (d + 1) * EPS * (np.abs(b) @ np.abs(x64).T + np.abs(y64)[None, :])
    bound = w * np.sum(2 * np.abs(r) * e + e * e + 5 * EPS * r * r, 1) + 1e-12 * np.abs(ref)
    for prec, tol in ((_lib.BH_GLM_FP32, bound), (_lib.BH_GLM_FP64, 1e-12 * (np.abs(ref) + N))):
        got = sf.log_density(pts, prec)
        assert np.all(np.abs(got - ref) <= tol), (prec, np.max(np.abs(got - ref) / tol))
    sf.release()
    fac.release()
