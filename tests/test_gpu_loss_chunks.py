"""The loss passes at the sizes where their split changes (needs a gfx950 GPU): images of one
pixel, one row or one column, chunks of two rows with a last chunk of one, strips that end
inside a workgroup's 256 row elements, and images tall enough for long chunks.  The gradient
is the reference's bit for bit whatever the split.  The loss value is a sum in an unspecified
order: a lane sums at most 32 terms, a tree 256 lanes, the workgroups in binary64, so each mean
is within (32 + 8 + 4) 2^-24 = 2.6e-6 of itself of the binary64 sum of the same terms; the
means are below 0.3 here (L1) and 1 (SSIM, weighed 0.2), so 2e-6 covers the loss."""
import numpy as np
import pytest

import oracle_lib as O
from splatrs_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("width,height", [(1, 1), (1, 23), (40, 1), (85, 3), (86, 11), (257, 95),
                                          (700, 477), (5, 3001), (1400, 950)])
def test_loss_split(ctx, width, height):
    print(f"[gpu-case] photometric loss {width}x{height}", flush=True)
    rng = np.random.default_rng(width * 10007 + height)
    x = rng.uniform(0, 1, (height, width, 3)).astype(np.float32)
    y = np.clip(x + rng.normal(0, 0.1, x.shape), 0, 1).astype(np.float32)
    loss, grad = ctx.photometric_loss(x, y, width, height, 0.2)
    _, go = O.photometric_loss(x, y, width, height, 0.2)
    assert np.array_equal(grad.view(np.uint32), go.view(np.uint32))
    ssim, l1 = O.loss_sums64(x, y, width, height)
    want = 0.8 * l1 / x.size + 0.2 * (1.0 - ssim / x.size)
    assert abs(loss - want) <= 2e-6
