"""What a half-step writes: of records too wide to stage in LDS only those that
moved, with a sample of them copied, and of small ones none where none moved."""
import numpy as np
import pytest
import torch

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu

CONSTANT = """
inline REAL constant_logpdf(const uint data_len, const uint params_len, const REAL* params, const uint dim,
                            const REAL* x) {
    return params[0];
}
"""


@pytest.mark.parametrize("wgs,dim", [(256, 48), (512, 32)])
def test_unmoved_records_are_not_written(wgs, dim):
    """A log density of 0 everywhere accepts some 60% of the proposals, one of
    minus infinity none: of three record's lengths (own, partner's, written) a
    half-step then moves two.  The half-way point between those shares, 1 and
    2 / 2.6 = 0.77, is 0.88."""
    fac = engine.HipBayaderaFactory(0, wgs)
    m = models.distribution_model(CONSTANT, "constant", dimension=dim, params_size=1)
    sf = fac.mcmc_factory(m)
    ms = []
    for value in (0.0, float("-inf")):
        s = sf.create_sampler(3, 1 << 19, [value]).set_exec(_lib.BH_EXEC_STEPWISE).set_timing(True)
        s.init_position(4, [-1, 1] * dim)
        runs = []
        for _ in range(6):
            s.burn_in(20, 2.0)
            runs.append(s.last_gpu_ms())
        ms.append(min(runs))
        s.release()
    assert ms[1] < 0.88 * ms[0], ms
    sf.release()
    fac.release()


def test_sample_of_records_too_wide_to_stage():
    """A step moves 2.15 record's lengths (own, partner's, those of the 15% that
    move), a sample two more where the ensemble is copied: 1.93 times as much."""
    dim, walkers = 48, 1 << 19
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.diag_gaussian_model(dim))
    s = sf.create_sampler(3, walkers, [0.0] * dim + [1.0] * dim).set_exec(_lib.BH_EXEC_STEPWISE).set_timing(True)
    s.init_position(4, [-2, 2] * dim)
    s.burn_in(20, 2.0)
    out = torch.empty(4 * walkers, dim, device="cuda")
    steps, samples = [], []
    for _ in range(6):
        s.burn_in(20, 2.0)
        steps.append(s.last_gpu_ms() / 20)
        s.sample(4 * walkers, out=out)
        samples.append(s.last_gpu_ms() / 4)
    assert min(samples) < 1.93 * min(steps), (samples, steps)
    assert np.array_equal(out[3 * walkers:].cpu().numpy(), s.state()[0].reshape(walkers, dim))
    s.release()
    sf.release()
    fac.release()


def test_small_records_are_not_written_where_none_moved():
    """Seven coordinates: 32 bytes are read and at most written for a walker and
    its log density, and one line of 128 for its partner: 192 and, with none
    moved, 160, which is 0.83.  Half-way to 1 is 0.92."""
    dim = 7
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.distribution_model(CONSTANT, "constant", dimension=dim, params_size=1))
    ms = []
    for value in (0.0, float("-inf")):
        s = sf.create_sampler(3, 1 << 22, [value]).set_timing(True)
        s.init_position(4, [-1, 1] * dim)
        runs = []
        for _ in range(6):
            s.burn_in(20, 2.0)
            runs.append(s.last_gpu_ms())
        ms.append(min(runs))
        s.release()
    assert ms[1] < 0.92 * ms[0], ms
    sf.release()
    fac.release()
