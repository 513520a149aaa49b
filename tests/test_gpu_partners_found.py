"""Half-steps of large ensembles of small records, whose partners are found
beforehand: the smallest and largest halves that take that path, partial tiles
and regions, both partner modes, against the oracle."""
import numpy as np
import pytest

import oracle as O
from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu

FLAT, WALKER = _lib.BH_PARTNER_FLAT, _lib.BH_PARTNER_WALKER


@pytest.mark.parametrize("wgs,half,partner", [
    (256, 1 << 22, FLAT), (256, (1 << 22) + 5 * 256, WALKER), (64, (1 << 22) + 8192 + 64, FLAT),
    (1024, (1 << 23) - 1024, WALKER), (256, (1 << 23) + 256, FLAT), (256, 1 << 25, WALKER)])
def test_one_coordinate(wgs, half, partner):
    """The uniform density takes no transcendental function: the same bits."""
    fac = engine.HipBayaderaFactory(0, wgs)
    sf = fac.mcmc_factory(models.uniform_model())
    s = sf.create_sampler(7, 2 * half, [-1, 2]).set_partner(partner)
    s.init(7)
    s.init_position(3, [-1, 2])
    ref = O.Stretch(O.UNIFORM_LOGPDF, 1, 2 * half, [-1, 2], 7, params_len=2, wgs=wgs, partner=partner,
                    threads=16)
    ref.init(7)
    ref.init_position(3, [-1, 2])
    s.move_bare()
    ref.move_bare()
    x = s.sample()
    assert np.array_equal(x, ref.sample())
    assert np.array_equal(s.state()[0].reshape(-1), ref.xs)
    s.release()
    sf.release()
    fac.release()


@pytest.mark.parametrize("half,partner", [
    (1 << 22, WALKER), ((1 << 22) + 256, FLAT), ((1 << 22) + 8192 - 256, WALKER), (1 << 24, FLAT)])
def test_two_coordinates(half, partner):
    """Independent Gaussians; a log density's last bit moves an accept test now
    and then, another partner would move every third walker."""
    params = np.array([0.5, -1.0, 2.0, 0.5], np.float32)
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.diag_gaussian_model(2))
    s = sf.create_sampler(9, 2 * half, params).set_partner(partner)
    s.init(9)
    s.init_position(4, [-3, 3, -3, 3])
    ref = O.Stretch(O.DIAG_GAUSS_LOGPDF, 2, 2 * half, params, 9, params_len=4, partner=partner, threads=16)
    ref.init(9)
    ref.init_position(4, np.array([[-3, 3], [-3, 3]], np.float32))
    for _ in range(2):
        s.move_bare()
        ref.move_bare()
    same = np.all(s.state()[0].reshape(-1, 2) == ref.xs.reshape(-1, 2), axis=1).mean()
    assert same > 0.995, same
    s.release()
    sf.release()
    fac.release()
