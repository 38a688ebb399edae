"""The scorer's packed matrix operands after Adam rewrote them (needs a gfx950 GPU): they are
those of a scorer created from the same weights, so both give the same logits and the same
gradient, bit for bit; batches of one chunk, several, and a number that leaves rows over."""
import numpy as np
import pytest

from splatrs_amd import abi
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 64, 1000, 1088, 20000])
def test_operands_follow_the_weights(batch):
    print(f"[gpu-case] scorer operands batch={batch}", flush=True)
    ctx = abi.Context(0)
    rng = np.random.default_rng(batch)
    n = 3 * batch
    p = (rng.normal(0, 1, rec.SCORER_PARAMS) * 0.25).astype(np.float32)
    x = rng.normal(0, 1, (n, 12)).astype(np.float32)
    y = rng.integers(0, 8, n).astype(np.uint8)
    w = rng.uniform(0.5, 2.0, n).astype(np.float32)
    a = abi.Scorer(ctx, p)
    a.fit(x, y, w, rec.scorer_fit_config(epochs=1, batch=batch, lr=0.1, seed=2))
    assert (a.params() != p).sum() > 9000
    b = abi.Scorer(ctx, a.params())
    assert np.array_equal(a.forward(x), b.forward(x))
    (la, ga), (lb, gb) = a.loss_grad(x, y, w), b.loss_grad(x, y, w)
    assert la == lb and np.array_equal(ga, gb)
    a.close()
    b.close()
    ctx.close()
