"""Work-groups that run a pair of problems give every problem what a small
batch, one problem to a work-group, gives it: bit for bit."""

import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fac():
    f = engine.HipBayaderaFactory(0, 256)
    yield f
    f.release()


def _run(fac, G, dims, params, hyper, lim, W, where, partner, seed):
    bt = fac.batch(models.hbb_model(G), params, dims, hyper, W).set_partner(partner).set_state(where)
    bt.init_position(17 + seed, lim)
    bt.burn_in(5 + 2 * seed, 2, 2.0)
    ser = np.zeros(3 * int(np.sum(dims)), np.float32)
    r = bt.run(9 + 2 * seed, 3, 2.0, series=ser)
    xs, lf = bt.state()
    out = [(xs[b], lf[b], r["acceptance-rate"][b], r["mean"][b], r["sd"][b]) for b in range(len(dims))]
    return out, bt.series_blocks(ser, 3)


# more problems than go round at once (odd and even counts, all dimensions up
# to the model's, more coordinates than threads), state in global memory and in
# LDS
@pytest.mark.parametrize("W,G,B,where,partner", [
    (128, 50, 3333, _lib.BH_BATCH_STATE_GLOBAL, _lib.BH_PARTNER_FLAT),
    (256, 50, 1400, _lib.BH_BATCH_STATE_GLOBAL, _lib.BH_PARTNER_WALKER),
    (128, 100, 1501, _lib.BH_BATCH_STATE_GLOBAL, _lib.BH_PARTNER_FLAT),
    (128, 30, 2047, _lib.BH_BATCH_STATE_LDS, _lib.BH_PARTNER_FLAT),
])
def test_pairs_equal_single(fac, W, G, B, where, partner):
    rng = np.random.default_rng(B)
    groups = rng.integers(1, G + 1, B)
    groups[:3] = 1, G, G // 2
    params, dims = [], []
    for g in groups:
        n = rng.integers(5, 200, g)
        params.append(np.concatenate([n, rng.binomial(n, 0.3), [1.5]]).astype(np.float32))
        dims.append(int(g) + 2)
    hyper = [1] * B
    lim = np.zeros((B, G + 2, 2), np.float32)
    lim[:, :, 0], lim[:, :, 1] = -1.0, 1.0
    got, gs = _run(fac, G, dims, params, hyper, lim, W, where, partner, 0)
    for first in (0, B - 50):
        s = slice(first, first + 50)
        want, ws = _run(fac, G, dims[s], params[s], hyper[s], lim[s], W, where, partner, first)
        for a, b in zip(got[s], want):
            assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b))
        assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(gs[s], ws))
