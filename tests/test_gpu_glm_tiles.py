"""Edges of the likelihood kernels' tiles: rows around the 16-row blocks, the
row ranges and the work-group that adds them up, features around the padded
16, 32 and 64, points that do and do not fill a launch."""
import numpy as np
import pytest

import oracle as O
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


# ranges fewer than, equal to and more than a point's threads (WGS / 16)
@pytest.mark.parametrize("wgs", [64, 256, 1024])
@pytest.mark.parametrize("N,d", [(40, 32), (1100, 64), (9001, 32)])
def test_logistic_range_sums(wgs, N, d):
    """fp64 log posteriors: every sum in double, 1e-12 of the terms' size."""
    rng = np.random.default_rng([N, d, wgs])
    X = models.to_bf16(rng.standard_normal((N, d)).astype(np.float32) / np.sqrt(d)).reshape(N, d)
    y = (rng.random(N) < 0.5).astype(np.float32)
    pts = rng.standard_normal((300, d)).astype(np.float32)
    fac = engine.HipBayaderaFactory(0, wgs)
    sf = fac.mcmc_factory(models.glm_logistic_model(X, y, 5.0))
    got = sf.log_density(pts, _lib.BH_GLM_FP64)
    eta = pts.astype(np.float64) @ models.from_bf16(X).reshape(N, d).astype(np.float64).T
    ref = eta @ y - np.sum(np.logaddexp(0.0, eta), 1) - 0.5 * np.sum(pts.astype(np.float64) ** 2, 1) / 25.0
    assert np.all(np.abs(got - ref) <= 1e-12 * (np.sum(np.abs(eta), 1) + N + 1))
    sf.release()
    fac.release()


@pytest.mark.parametrize("wgs,walkers", [(256, 512), (256, 1536), (1024, 2048)])
def test_screened_chain_equals_fp64_chain(wgs, walkers):
    """The guarded chain decides as the fp64 one, whatever work-group screens
    it: the same positions and accounting."""
    N, d = 3001, 32
    rng = np.random.default_rng(3)
    X = models.to_bf16(rng.standard_normal((N, d)).astype(np.float32) / np.sqrt(d)).reshape(N, d)
    beta = rng.standard_normal(d)
    eta = models.from_bf16(X).reshape(N, d).astype(np.float64) @ beta
    y = (rng.random(N) < 1.0 / (1.0 + np.exp(-eta))).astype(np.float32)
    fac = engine.HipBayaderaFactory(0, wgs)
    sf = fac.mcmc_factory(models.glm_logistic_model(X, y, 5.0))
    lim = np.stack([beta - 0.3, beta + 0.3], 1)
    out = []
    for prec, guard in ((_lib.BH_GLM_FP64, 0.0), (_lib.BH_GLM_FP16X2, 2e-3), (_lib.BH_GLM_FP16, 6e-3)):
        s = sf.create_sampler(5, walkers, np.zeros(1, np.float32))
        s.set_glm_precision(prec).set_partner(_lib.BH_PARTNER_WALKER)
        if guard:
            s.set_glm_guard(guard)
        s.init_position(6, lim)
        s.burn_in(6, 2.0)
        s.init_move(2.0, 5)
        for _ in range(5):
            s.move()
        out.append((s.state()[0], *s.read_accounting(5)))
        s.release()
    for o in out[1:]:
        for x, w in zip(o, out[0]):
            assert np.array_equal(x, w)
    sf.release()
    fac.release()


def test_logistic_matches_oracle_at_one_row():
    X = models.to_bf16(np.full((1, 32), 0.25, np.float32)).reshape(1, 32)
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.glm_logistic_model(X, np.ones(1, np.float32), 5.0))
    pts = np.linspace(-2, 2, 5 * 32).reshape(5, 32).astype(np.float32)
    ref = O.glm_logpost(models.from_bf16(X).reshape(1, 32), np.ones(1, np.float32), 5.0, pts)
    assert np.allclose(sf.log_density(pts, _lib.BH_GLM_FP64), ref, rtol=1e-12, atol=1e-12)
    sf.release()
    fac.release()
