"""Sorted partners of records of two coordinates, bit for bit against the oracle:
records that run on past a region's end, the wrap from the last element to the
first, and the last partial tile."""
import numpy as np
import pytest

import oracle as O
from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu

FLAT, WALKER = _lib.BH_PARTNER_FLAT, _lib.BH_PARTNER_WALKER
TILE = 8192  # walkers


def partner_offsets(seed, odd_or_even, half, partner):
    """First elements of the partners of a half-step of step 0 (the draws of
    amd-gcn-mcmc-stretch.cl:46-57), in numpy."""
    c = [np.arange(half, dtype=np.uint64), np.full(half, 0, np.uint64), np.full(half, odd_or_even, np.uint64),
         np.full(half, 0xBEEFF00D, np.uint64)]
    k, low = [seed, 0xDECAFBAD], np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        s = np.uint64(32)
        c = [(p1 >> s) ^ c[1] ^ np.uint64(k[0]), p1 & low, (p0 >> s) ^ c[3] ^ np.uint64(k[1]), p0 & low]
        k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
    u = (np.float32(0.5) + (c[0] >> np.uint64(9)).astype(np.float32)) * np.float32(2.0 ** -23)
    if partner == WALKER:
        return np.minimum((u * np.float32(half)).astype(np.uint32), half - 1) * 2
    e = ((u * np.float32(half)) * np.float32(2)).astype(np.uint32)
    return np.where(e >= 2 * half, e - 2 * half, e)


@pytest.mark.parametrize("half,partner,seed", [
    (1 << 22, FLAT, 1), (1 << 22, WALKER, 9), ((1 << 22) + 256, FLAT, 1), ((1 << 22) + TILE - 256, WALKER, 9),
    (1 << 23, FLAT, 1), (1 << 24, FLAT, 1)])
def test_against_the_oracle(half, partner, seed):
    """The uniform density of the first coordinate takes no transcendental
    function: positions are the same bits.  The draws of the first half-step
    include the last element of regions and of the half (of 2^24 walkers they
    are even elements only)."""
    if partner == FLAT and half < 1 << 24:
        e = partner_offsets(seed, 3333, half, partner)
        assert np.count_nonzero((e + 1) % (1 << 15) == 0) >= 50  # regions of 2^15 floats
        assert e.max() == 2 * half - 1
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.distribution_model(models.UNIFORM_SOURCE, name="uniform", dimension=2, params_size=2))
    s = sf.create_sampler(seed, 2 * half, [-1, 2]).set_partner(partner).init_position(3, [-1, 2, -5, 5])
    ref = O.Stretch(O.UNIFORM_LOGPDF, 2, 2 * half, [-1, 2], seed, params_len=2, partner=partner, threads=16)
    ref.init_position(3, np.array([[-1, 2], [-5, 5]], np.float32))
    for _ in range(2):
        s.move_bare()
        ref.move_bare()
        x, lf, _ = s.state()
        assert np.all(lf == lf[0]) and np.isfinite(lf[0])
        want = ref.xs.reshape(-1, 2)
        for h in range(2):  # the last partial tile of each half by itself, then all
            tail = slice(h * half + half // TILE * TILE, (h + 1) * half)
            assert np.array_equal(x[tail], want[tail])
        assert np.array_equal(x, want)
    for h in (s, sf, fac):
        h.release()
