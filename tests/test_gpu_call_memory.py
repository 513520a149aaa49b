"""Results that land through pinned memory, through a copy, or in place: the
same values on either side of the size that divides them, and from several
threads that share a context's buffers."""

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from bayadera_amd import engine, models

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fac():
    f = engine.HipBayaderaFactory(0, 256)
    yield f
    f.release()


# 256 KB of results is the largest that is written into pinned memory; 64 MB
# the largest device block that is kept
@pytest.mark.parametrize("n", [4, 1024, 65532, 65536, 65540, 1 << 20, (1 << 24) + 4])
def test_host_and_device_results(fac, n):
    e = fac.direct_sampler_engine(models.gaussian_model())
    d = torch.empty(n, dtype=torch.float32, device="cuda")
    e.sample(7, [1.0, 2.0], n, out=d)
    for _ in range(2):  # a new block, then a kept one
        assert np.array_equal(e.sample(7, [1.0, 2.0], n), d.cpu().numpy())


@pytest.mark.parametrize("problems", [1, 3, 257, 4099])
def test_batch_results(fac, problems):
    """Means and deviations of one step equal those of the positions it left,
    to 128 float roundings of values of about 2."""
    rng = np.random.default_rng(problems)
    dims = rng.integers(1, 8, problems)
    params = [np.concatenate([np.zeros(d), np.eye(d).reshape(-1)]).astype(np.float32) for d in dims]
    bt = fac.batch(models.mvn_model(7), params, list(dims), [0] * problems, 128)
    lim = np.zeros((problems, 7, 2), np.float32)
    lim[:, :, 0], lim[:, :, 1] = -2.0, 2.0
    bt.init_position(11, lim)
    r = bt.run(5, 1, 2.0)
    xs, _ = bt.state()
    assert np.all((r["acceptance-rate"] >= 0) & (r["acceptance-rate"] <= 1))
    assert np.all(r["acceptance-rate"] * 128 == np.round(r["acceptance-rate"] * 128))
    for p, d in enumerate(dims):
        x = xs[p].astype(np.float64)
        assert np.allclose(r["mean"][p, :d], x.mean(0), rtol=0, atol=2e-5)
        assert np.allclose(r["sd"][p, :d], x.std(0), rtol=0, atol=2e-5)
        assert np.all(r["mean"][p, d:] == 0) and np.all(r["sd"][p, d:] == 0)


def test_threads_share_the_buffers(fac):
    rng = np.random.default_rng(3)
    data = [rng.standard_normal((4000 + 997 * i, 3)).astype(np.float32) for i in range(8)]
    de = fac.dataset_engine()

    def work(a):
        h = de.histogram(a)
        return h.limits, h.pdf, h.bin_ranks, de.data_mean(a), de.data_variance(a)

    alone = [work(a) for a in data]
    with ThreadPoolExecutor(4) as ex:
        for got, want in zip(ex.map(work, data * 4), alone * 4):
            assert all(np.array_equal(g, w) for g, w in zip(got, want))
