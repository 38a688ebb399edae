"""The order in which the scorer's gradient is summed (needs a gfx950 GPU).  64 samples make one
partial gradient, and the partial gradients are added one after the other, so a batch's gradient
is exactly the running binary32 sum of its 64-sample parts.  The scale 1/n of a part is a power
of two times the batch's: all products and roundings scale with it, exactly."""
import numpy as np
import pytest

from splatrs_amd import abi
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 256, 1024])
def test_partial_gradients_in_order(n):
    print(f"[gpu-case] scorer gradient of {n} samples", flush=True)
    ctx = abi.Context(0)
    rng = np.random.default_rng(n)
    p = (rng.normal(0, 1, rec.SCORER_PARAMS) * 0.25).astype(np.float32)
    x = rng.normal(0, 1, (n, 12)).astype(np.float32)
    y = rng.integers(0, 8, n).astype(np.uint8)
    w = rng.uniform(0.5, 2.0, n).astype(np.float32)
    s = abi.Scorer(ctx, p)
    loss, grad = s.loss_grad(x, y, w)
    want_loss, want = np.float32(0.0), np.zeros(rec.SCORER_PARAMS, np.float32)
    for k in range(0, n, 64):
        part_loss, part = s.loss_grad(x[k:k + 64], y[k:k + 64], w[k:k + 64])
        want = want + np.float32(64 / n) * part
        want_loss = want_loss + np.float32(64 / n) * np.float32(part_loss)
    s.close()
    ctx.close()
    assert np.array_equal(grad.view(np.uint32), want.astype(np.float32).view(np.uint32))
    assert np.float32(loss) == want_loss
