"""A sample written by its last moves equals the ensemble it leaves, and a
copied one (a part of an ensemble, an output that is not 16-byte aligned)."""

import numpy as np
import pytest
import torch

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("partner", [_lib.BH_PARTNER_FLAT, _lib.BH_PARTNER_WALKER])
@pytest.mark.parametrize("wgs,dim,walkers", [(256, 1, 512), (64, 3, 1280), (256, 8, 512), (256, 9, 1536),
                                             (256, 32, 512), (1024, 4, 2048), (1024, 16, 4096)])
def test_samples(wgs, dim, walkers, partner):
    fac = engine.HipBayaderaFactory(0, wgs)
    mf = fac.mcmc_factory(models.diag_gaussian_model(dim))
    rng = np.random.default_rng(dim)
    params = np.concatenate([rng.standard_normal(dim), rng.uniform(0.5, 2.0, dim)]).astype(np.float32)
    lim = np.tile(np.array([-3.0, 3.0], np.float32), (dim, 1))

    def sampler():
        s = mf.create_sampler(7, walkers, params)
        s.set_partner(partner).set_exec(_lib.BH_EXEC_STEPWISE)
        s.init_position(3, lim)
        return s

    n = walkers * 2 + 5
    raw = torch.empty(n * dim + 1, dtype=torch.float32, device="cuda")
    got = []
    for o in (raw[:n * dim], raw[1:]):  # the second is not 16-byte aligned
        s = sampler()
        s.sample(n, out=o.view(n, dim))
        got.append(o.clone().cpu().numpy().reshape(n, dim))
        s.release()
    s = sampler()
    one = s.sample(walkers)
    assert np.array_equal(one, s.state()[0].reshape(walkers, dim))
    assert np.array_equal(got[0], got[1])
    assert np.array_equal(got[0][:walkers], one)
    two = s.sample(walkers)
    assert np.array_equal(got[0][walkers:2 * walkers], two)
    assert np.array_equal(got[0][2 * walkers:], s.sample(5))
    s.release()
    mf.release()
    fac.release()
