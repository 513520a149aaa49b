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
