"""Contraction units cut into pieces: a problem's log posteriors do not depend
on the pieces its rows are cut into, only their double sums' order does."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fac():
    f = engine.HipBayaderaFactory(0, 256)
    yield f
    f.release()


def _problem(rng, n, d):
    codes = rng.integers(0, 120, (n, d)).astype(np.uint8) | (rng.integers(0, 2, (n, d)) << 7).astype(np.uint8)
    return codes, (rng.uniform(0.5, 2.0, d) / 448 / np.sqrt(d)).astype(np.float32), (rng.random(n) < 0.5).astype(np.float32)


# rows around the pieces' edges, one and several runs of 2048 rows, a last run
# of one row; with much other work (long pieces) and alone (short ones)
@pytest.mark.parametrize("prec", [_lib.BH_GLM_FP16X2, _lib.BH_GLM_BF16X3, _lib.BH_GLM_FP32, _lib.BH_GLM_FP64])
def test_pieces_do_not_change_the_sums(fac, prec):
    rng = np.random.default_rng(1)
    W = 512
    shapes = [(n, d) for n in (1, 255, 256, 383, 384, 385, 2048, 2049, 2431, 2433, 6000) for d in (5, 40)]
    shapes += [(60000, 32)] * 6 + [(60000, 64)] * 6
    probs = [_problem(rng, n, d) for n, d in shapes]
    lim = np.zeros((len(probs), 64, 2), np.float32)
    lim[:, :, 0], lim[:, :, 1] = -1.0, 1.0

    def lp(which):
        m = models.GlmBatchModel(*[list(v) for v in zip(*[probs[i] for i in which])], 5.0)
        bt = fac.glm_batch(m, W).set_precision(prec)
        bt.init_position(9 + which[0], lim[which])
        return bt.log_density(prec)

    together = lp(list(range(len(probs))))
    for i, (n, d) in enumerate(shapes[:23]):
        alone = lp([i])[0]
        # every term is at most |eta| + 1, summed in double in another order
        assert np.allclose(together[i], alone, rtol=1e-13, atol=1e-13 * n * 64)
