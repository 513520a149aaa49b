"""Linear regression data: larger than 2^32 padded floats, and in device memory
that other work is still writing."""
import numpy as np
import pytest
import torch

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def test_rows_past_2p32_floats():
    """2^28 rows, padded from 1 to 16 columns: 17 GB.  The bound is that of the
    tiles' test (test_gpu_glm_tiles.py) for one feature; the sum over rows is
    in double."""
    N, d = 1 << 28, 1
    i = torch.arange(N, device="cuda")
    x = ((i * 7919 + 13) % 1021 - 510).to(torch.float32) / 256
    y = 0.75 * x + ((i * 104729 + 5) % 4093 - 2046).to(torch.float32) / 8192
    del i
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.glm_gaussian_model(x.cpu().numpy().reshape(N, d), y.cpu().numpy(), 10.0, 1.0))
    pts = np.array([[0.75, -1.5], [-0.5, 0.25]], np.float32)
    got = {p: sf.log_density(pts, p) for p in (_lib.BH_GLM_FP32, _lib.BH_GLM_FP64)}
    for k, (b, ls) in enumerate(pts.astype(np.float64)):
        r = y.double() - b * x.double()
        w = 0.5 * np.exp(-2 * ls)
        ref = -N * (ls + 0.5 * np.log(2 * np.pi)) - w * float((r * r).sum()) - 0.5 * (b * b / 100.0 + ls ** 2)
        e = (d + 1) * EPS * (abs(b) * x.double().abs() + y.double().abs())
        bound = w * float((2 * r.abs() * e + e * e + 5 * EPS * r * r).sum()) + 1e-12 * abs(ref)
        assert abs(got[_lib.BH_GLM_FP32][k] - ref) <= bound
        assert abs(got[_lib.BH_GLM_FP64][k] - ref) <= 1e-12 * (abs(ref) + N)
        del r, e
    sf.release()
    fac.release()


def test_data_that_the_default_stream_is_writing():
    """X and y on the device, written behind some 50 ms of other work: the same
    log posteriors as from host copies, bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn(5000, 7, generator=g, device="cuda")
    y = torch.randn(5000, generator=g, device="cuda")
    pts = np.random.default_rng(4).standard_normal((40, 8)).astype(np.float32)
    fac = engine.HipBayaderaFactory(0, 256)
    out = []
    for device in (False, True):
        Xd, yd = torch.zeros_like(X), torch.zeros_like(y)
        torch.cuda.synchronize()
        torch.cuda._sleep(100_000_000)
        Xd.copy_(X)
        yd.copy_(y)
        data = (Xd, yd) if device else (Xd.cpu().numpy(), yd.cpu().numpy())
        sf = fac.mcmc_factory(models.GlmModel("gaussian", *data, 10.0))
        out.append([sf.log_density(pts, p) for p in (_lib.BH_GLM_FP32, _lib.BH_GLM_FP64)])
        sf.release()
    assert np.array_equal(out[0], out[1])
    fac.release()
