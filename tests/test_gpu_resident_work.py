"""What the resident steps work with: draws that were never made are not used,
chunk buffers are the context's and not a sampler's."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu

# as many rounds as the coordinate says, at most 2^20 (some ms of one thread)
ROUNDS = """
inline REAL rounds_logpdf(const uint data_len, const uint params_len, const REAL* params, const uint dim,
                          const REAL* x) {
    const uint n = (uint)fmin(fabs(x[0]), 1048576.0f);
    REAL t = 0.0f;
    for (uint i = 0; i < n; i++) t = t * params[0] + x[0];
    return -0.5f * x[0] * x[0] - 1e-6f * t;
}
"""


@pytest.mark.parametrize("wgs,walkers,steps", [(64, 1024, 5), (64, 2176, 4)])
def test_density_past_the_last_half_step(wgs, walkers, steps):
    """An odd number of steps leaves half of a round, 1088 walkers to a half 64
    threads without one.  The buffers a context used before hold 1e9 in every
    float: a density taken at those would run 2^20 rounds (over 2 ms; the steps
    themselves take some 20 us)."""
    fac = engine.HipBayaderaFactory(0, wgs)
    sf = fac.mcmc_factory(models.distribution_model(ROUNDS, "rounds", dimension=1, params_size=1))
    de = fac.dataset_engine()
    out = []
    for mode in (_lib.BH_EXEC_STEPWISE, _lib.BH_EXEC_AUTO):
        s = sf.create_sampler(3, walkers, [0.5]).set_exec(mode).set_timing(True)
        s.init_position(4, [-3, 3])
        s.burn_in(steps, 2.0)
        for e in range(10, 23):  # a kept block of every size, full of 1e9
            de.data_mean(np.full((1 << e, 1), 1e9, np.float32))
        s.burn_in(steps, 2.0)
        ms = s.last_gpu_ms()
        out.append(s.state())
        s.release()
    assert all(np.array_equal(x, y) for x, y in zip(*out))
    assert ms < 1.0, ms
    sf.release()
    fac.release()


def test_fresh_samplers_share_the_chunk_buffers():
    """A second sampler's job takes no device memory of its own: 1024 walkers x
    4 draw 16 MiB and trace 8 MiB per chunk."""
    import torch
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.diag_gaussian_model(4))
    params = np.array([0, 0, 0, 0, 1, 1, 1, 1], np.float32)

    def sampler(seed):
        return sf.create_sampler(seed, 1024, params).init_position(seed, [-2, 2] * 4)

    def job(s):
        s.burn_in(256, 2.0)
        s.run_sampler(1024, 2.0)
        s.sample(1 << 18, out=torch.empty(1 << 18, 4, device="cuda"))

    first, second = sampler(1), sampler(2)
    job(first)  # the context's buffers, and torch's block for the draws
    second.init_move(2.0, 1024)  # the sums of this many steps are the sampler's own
    before = torch.cuda.mem_get_info()[0]
    job(second)
    assert torch.cuda.mem_get_info()[0] == before
    for h in (first, second, sf, fac):
        h.release()


@pytest.mark.parametrize("walkers,fewest", [(1024, 2), (4096, 3), (8192, 4)])
def test_calls_of_few_steps(walkers, fewest):
    """Calls of fewer steps take the two launches of each step, longer ones one
    launch, and a resident sampler always one."""
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.diag_gaussian_model(2))
    s = sf.create_sampler(3, walkers, [0, 0, 1, 1]).init_position(4, [-2, 2] * 2)
    for n in (1, 2, 3, 4):
        for mode, launches in ((_lib.BH_EXEC_AUTO, 1 if n >= fewest else 2 * n), (_lib.BH_EXEC_RESIDENT, 1)):
            if mode == _lib.BH_EXEC_RESIDENT and walkers > 4096:
                continue  # refused
            s.set_exec(mode).set_kernel_timing(True)
            s.burn_in(n, 2.0)
            assert s.kernel_timing()["launches"] == launches
    for h in (s, sf, fac):
        h.release()


@pytest.mark.parametrize("wgs", [64, 256])
@pytest.mark.parametrize("dim,walkers", [(1, 512), (9, 1024), (38, 1024), (2, 2560), (1, 12288), (4, 7168), (7, 4096)])
def test_ensembles_that_run_resident(wgs, dim, walkers):
    """By themselves, all their steps in one launch, also where RESIDENT is
    refused (the ensembles of test_gpu_resident.py among them)."""
    fac = engine.HipBayaderaFactory(0, wgs)
    sf = fac.mcmc_factory(models.diag_gaussian_model(dim))
    s = sf.create_sampler(3, walkers, [0.0] * dim + [1.0] * dim).init_position(4, [-2, 2] * dim)
    s.set_kernel_timing(True)
    s.burn_in(9, 2.0)
    assert s.kernel_timing()["launches"] == 1
    for h in (s, sf, fac):
        h.release()
