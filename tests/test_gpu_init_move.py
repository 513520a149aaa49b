"""init-move! where its buffers cannot be made."""
import numpy as np
import pytest

from bayadera_amd import _lib, engine, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1 << 44, (1 << 62) + 1])
def test_no_move_after_one_that_failed(steps):
    """The sums of 2^44 steps are more than any device holds, those of 2^62 + 1
    more than 64 bits count: refused, and so is the move after the former; the
    next init-move! is as on a sampler that saw none of it."""
    fac = engine.HipBayaderaFactory(0, 256)
    sf = fac.mcmc_factory(models.diag_gaussian_model(2))
    a, b = (sf.create_sampler(3, 1024, [0, 0, 1, 1]).init_position(4, [-2, 2] * 2) for _ in range(2))
    a.init_move(2.0, 4).move()
    b.init_move(2.0, 4).move()
    with pytest.raises(_lib.BayaderaError):
        a.init_move(2.0, steps)
    if steps < 1 << 60:
        with pytest.raises(_lib.BayaderaError):
            a.move()
        with pytest.raises(_lib.BayaderaError):
            a.read_accounting(1)
    a.init_move(2.0, 4).move()
    b.init_move(2.0, 4).move()
    assert all(np.array_equal(x, y) for x, y in zip(a.read_accounting(1), b.read_accounting(1)))
    assert all(np.array_equal(x, y) for x, y in zip(a.state(), b.state()))
    for h in (a, b, sf, fac):
        h.release()
