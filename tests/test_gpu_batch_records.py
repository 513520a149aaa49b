"""Batched posteriors whose records are moved a lane to a record or as runs of a
wave's records, in LDS and in place: every problem is the oracle's single
sampler, bit for bit (the uniform density of the first coordinate takes no
transcendental function)."""
import numpy as np
import pytest

import oracle as O
from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu

FLAT, WALKER = _lib.BH_PARTNER_FLAT, _lib.BH_PARTNER_WALKER
LDS, GLOBAL = _lib.BH_BATCH_STATE_LDS, _lib.BH_BATCH_STATE_GLOBAL


def _batch(fac, dim, dims, walkers):
    m = models.distribution_model(models.UNIFORM_SOURCE, name="uniform", dimension=dim, params_size=2)
    return fac.batch(m, [np.array([-1, 2], np.float32)] * len(dims), dims, [2] * len(dims), walkers)


# the model's dimension decides the form in place, a problem's own in LDS; an
# odd number of problems leaves one without a pair
@pytest.mark.parametrize("dim,dims,walkers", [
    (1, [1, 1, 1], 128), (7, [1, 2, 3, 4, 5, 6, 7], 384), (8, [1, 7, 8], 128), (11, [3, 8, 9, 10, 11], 256),
    (12, [1, 5, 12], 128), (33, [1, 2, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33], 128), (66, [63, 64, 65, 66], 128)])
@pytest.mark.parametrize("where", [LDS, GLOBAL])
@pytest.mark.parametrize("partner", [FLAT, WALKER])
def test_against_the_oracle(dim, dims, walkers, where, partner):
    fac = engine.HipBayaderaFactory(0, 256)
    bt = _batch(fac, dim, dims, walkers).set_partner(partner)
    bt.set_state(where)
    lim = np.zeros((len(dims), dim, 2), np.float32)
    lim[:, :, 0], lim[:, :, 1] = -1.0, 2.0
    bt.init_position(100, lim)
    bt.burn_in(50, 5, 2.0)
    xs, _ = bt.state()
    for b, d in enumerate(dims):
        ref = O.Stretch(O.UNIFORM_LOGPDF, d, walkers, [-1, 2], 50 + 2 * b, wgs=64, params_len=2, partner=partner)
        ref.init_position(100 + b, lim[b, :d])
        ref.burn_in(5, 2.0)
        assert np.array_equal(xs[b], ref.xs.reshape(walkers, d)), d
    bt.release()
    fac.release()


def test_small_records_take_a_lane_each():
    """A run of eight passes costs one coordinate what it costs eight (0.83 of it
    was measured); a lane to a record 0.39 of it.  Half-way is 0.6."""
    fac = engine.HipBayaderaFactory(0, 256)
    ms = {}
    for d in (1, 8):
        bt = _batch(fac, d, [d] * 1000, 256)
        bt.set_state(LDS)
        lim = np.zeros((1000, d, 2), np.float32)
        lim[:, :, 0], lim[:, :, 1] = -1.0, 2.0
        bt.init_position(3, lim)
        runs = []
        for _ in range(5):
            bt.burn_in(5, 100, 2.0)
            runs.append(bt.last_gpu_ms())
        ms[d] = min(runs)
        bt.release()
    assert ms[1] < 0.6 * ms[8], ms
    fac.release()
