"""The loss is summed in 64 bits.  With all parameters zero the outputs are zero and the
differences are the targets, so the loss is known: to 1e-13 (sums of at most 200 terms
in a row, each rounded to 1.1e-16 of it) from chan_mlp_grad, to float's
rounding from chan_mlp_train.  Counts in one block and in many, with remainders."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 129, 8192, 8193, 40000, 65536])
def test_loss_in_64_bits(n):
    from channel_amd.closure import Mlp
    print("[case] loss", n, flush=True)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, mo.IN)).astype(np.float32)
    T = rng.standard_normal((n, mo.OUT)).astype(np.float32)
    want = np.sum(T.astype(np.longdouble) ** 2) / (6 * n)
    m = Mlp(n)
    m.set_params(np.zeros(mo.NPARAM, dtype=np.float32))
    m.set_data(X, T)
    loss, _ = m.grad(0, n)
    assert abs(loss - want) <= 1e-13 * want
    losses, _ = m.train(1, n, 1e-3)
    assert abs(losses[0] - want) <= 2e-7 * want  # the sum and its quotient, each rounded to a float
    m.close()
