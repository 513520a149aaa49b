"""Which ensembles have their partners sorted: those of densities that take few
parameters, while the memory for it is there."""
import numpy as np
import pytest
import torch

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu

LOOP = """
inline REAL loop_logpdf(const uint data_len, const uint params_len, const REAL* params, const uint dim,
                        const REAL* x) {
    REAL acc = 0.0f;
    for (uint i = 0; i < data_len; i++) acc -= (params[i] - x[0]) * (params[i] - x[0]);
    return acc * params[data_len];
}
"""


@pytest.mark.parametrize("values,is_sorted", [(0, True), (16, True), (32, False), (1000, False)])
def test_density_of_so_many_values(values, is_sorted):
    """2^23 walkers of one coordinate take 64 MiB (positions and log densities),
    and 16 bytes for each walker of a half where partners are sorted."""
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.distribution_model(LOOP, "loop", dimension=1, params_size=1))
    params = np.full(values + 1, 0.01, np.float32)
    sf.create_sampler(1, 512, params).release()
    before = torch.cuda.mem_get_info()[0]
    s = sf.create_sampler(3, 1 << 23, params)
    taken = before - torch.cuda.mem_get_info()[0]
    assert (taken > (64 << 20) + (32 << 20)) == is_sorted, taken
    for h in (s, sf, fac):
        h.release()


def test_buffers_given_back():
    """An allocation that fails takes the buffers (2^22 walkers to a half: 64 MiB),
    and the moves after it are those of a sampler that kept its own."""
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.uniform_model())
    a, b = (sf.create_sampler(7, 1 << 23, [-1, 2]).init_position(3, [-1, 2]) for _ in range(2))
    b.move_bare()
    b.move_bare()
    want = b.state()
    b.release()
    a.move_bare()
    before = torch.cuda.mem_get_info()[0]
    with pytest.raises(_lib.BayaderaError):
        a.init_move(2.0, 1 << 44)  # more than any device holds
    assert torch.cuda.mem_get_info()[0] - before >= 64 << 20
    a.move_bare()
    assert all(np.array_equal(x, y) for x, y in zip(a.state(), want))
    for h in (a, sf, fac):
        h.release()


def test_kernel_timing_of_sorted_steps():
    """Every half-step counts, and each with its half of the sort: every second
    or third one timed gives the average of all.  (The half that brought the sort
    along took 1.6 to 1.8 times the other; a spread of 10% is allowed for.)"""
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.uniform_model())
    s = sf.create_sampler(7, 1 << 23, [-1, 2]).init_position(3, [-1, 2])
    s.burn_in(20, 2.0)
    ms, launches = {}, {}
    for every in (1, 2, 3):
        s.set_kernel_timing(True, every)
        s.burn_in(30, 2.0)
        t = s.kernel_timing()
        ms[every], launches[every] = t["avg_ms"], t["launches"]
    assert launches[1] == 60 and launches[2] == 60 and launches[3] == 40
    assert all(abs(ms[e] / ms[1] - 1) < 0.1 for e in (2, 3)), ms
    for h in (s, sf, fac):
        h.release()
