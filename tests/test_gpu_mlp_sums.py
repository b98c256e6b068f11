"""The closure's training sums at the sample counts where their launches change: a tile
with one live sample, one block, fewer partials than the rows that are added at a
time, exactly as many (128), one more, all 512 blocks, a second tile for one wave only.

Bars: as for any count, the gradient 5e-3 (relative L2) against the oracle with BF16
operands (one rounding of a BF16 operand that falls the other way is 4e-3 of that
operand), the loss 1e-5.  The epoch loss of a training call with a step of length 0,
which the Adam kernel adds up, is the same loss."""
import numpy as np
import pytest

from diablo3_amd.closure import Mlp
from oracle import mlp as om
from test_gpu_mlp import setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 64, 65, 960, 8192, 8193, 32768, 32769, 33000])
def test_sums_match_oracle(n):
    print(f"gradient and losses, {n} samples", flush=True)
    p, X, T, norm = setup(n, 6)
    m = Mlp(p)
    m.set_norm(norm)
    m.set_data(X, T)
    lw = (1.0, 0.5)
    loss, g = m.grad(n, lw)
    lo, go = om.loss_grad(p, norm, X, T, lw, emulate=True)
    hist = m.train(epochs=2, batch=n, lr=0.0, seed=2, loss_w=lw)
    e = np.linalg.norm(g - go) / np.linalg.norm(go)
    print(f"gradient {e:.1e}, loss {abs(loss - lo) / lo:.1e}, epochs {np.abs(hist - lo).max() / lo:.1e}", flush=True)
    assert e <= 5e-3
    assert abs(loss - lo) <= 1e-5 * lo
    assert np.all(np.abs(hist - lo) <= 1e-5 * lo)
    assert np.array_equal(m.params[om.live_mask()], p[om.live_mask()])
