"""The resident steps (draws, steps and accounting as separate launches per
chunk) against the per-half-step kernels, which take the same arithmetic and
trees: equal bit for bit, so there is no tolerance."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu
FLAT, WALKER = _lib.BH_PARTNER_FLAT, _lib.BH_PARTNER_WALKER


@pytest.fixture(scope="module", params=[256, 64])
def fac(request):
    f = engine.HipBayaderaFactory(0, request.param)
    yield f
    f.release()


def _pair(fac, dim, walkers, partner):
    rng = np.random.default_rng([dim, walkers])
    params = np.concatenate([rng.standard_normal(dim), rng.uniform(0.5, 2.0, dim)]).astype(np.float32)
    sf = fac.mcmc_factory(models.diag_gaussian_model(dim))
    out = []
    # (by itself the engine chooses the resident steps for all of these, also
    # for ensembles that set_exec refuses as too large for 64 KB)
    resident = _lib.BH_EXEC_AUTO
    for mode in (_lib.BH_EXEC_STEPWISE, resident):
        s = sf.create_sampler(17, walkers, params).set_exec(mode).set_partner(partner)
        s.init_position(18, np.tile(np.array([-3.0, 3.0], np.float32), dim))
        out.append(s)
    return sf, out


def _same_state(a, b):
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x, y)


# one to three walkers per thread (the last with threads past the half), records
# of whole and of partial 16-byte pieces, and numbers of half-steps that do and
# do not fill the kernel's rounds of four
@pytest.mark.parametrize("dim,walkers", [(1, 512), (3, 512), (4, 1024), (7, 1536), (9, 1024),
                                         (2, 2560), (3, 3072), (1, 5120), (2, 4608),
                                         (1, 12288), (4, 7168)])
@pytest.mark.parametrize("partner", [FLAT, WALKER])
def test_resident_equals_stepwise(fac, dim, walkers, partner):
    sf, (a, b) = _pair(fac, dim, walkers, partner)
    for s in (a, b):
        s.burn_in(5, 2.0)
        s.anneal(lambda i: 7.0 - i, 6, 2.5)
    _same_state(a, b)
    ra, rb = a.run_sampler(53, 2.0), b.run_sampler(53, 2.0)
    assert ra["acceptance-rate"] == rb["acceptance-rate"]
    assert np.array_equal(ra["means"], rb["means"])
    for x, y in zip(a.read_accounting(53), b.read_accounting(53)):
        assert np.array_equal(x, y)
    _same_state(a, b)
    # a sample that ends inside an ensemble, and inside its first half
    for n in (1, 3 * walkers + 5, 2 * walkers + walkers // 2 + 3):
        assert np.array_equal(a.sample(n), b.sample(n))
    _same_state(a, b)
    for s in (a, b):
        s.release()
    sf.release()


def test_resident_runs_of_several_chunks(fac):
    """More steps than one chunk of draws holds (16 MiB at 2 x 512 draws of 16
    bytes per step: 1024 bare steps, fewer accounted ones)."""
    sf, (a, b) = _pair(fac, 1, 1024, FLAT)
    for s in (a, b):
        s.burn_in(2051, 2.0)
    _same_state(a, b)
    ra, rb = a.run_sampler(2100, 2.0), b.run_sampler(2100, 2.0)
    assert np.array_equal(ra["means"], rb["means"])
    assert ra["acceptance-rate"] == rb["acceptance-rate"]
    n = 2060 * 1024
    assert np.array_equal(a.sample(n), b.sample(n))
    for s in (a, b):
        s.release()
    sf.release()


def test_resident_sample_leaves_what_follows_alone():
    import torch
    f = engine.HipBayaderaFactory(0, 256)
    sf, (a, b) = _pair(f, 3, 1024, WALKER)
    got = []
    for s in (a, b):
        buf = torch.full((3 * 2000 + 64,), 7.0, device="cuda")
        torch.cuda.synchronize()
        # an output that is only 4-byte aligned
        s.sample(2000, out=buf[1:6001])
        got.append(buf.cpu().numpy())
        s.release()
    assert np.array_equal(got[0], got[1])
    assert got[1][0] == 7.0 and np.all(got[1][6001:] == 7.0)
    sf.release()
    f.release()
