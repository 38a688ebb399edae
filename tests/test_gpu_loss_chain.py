"""How many terms a lane of the loss passes adds in binary32 (needs a gfx950 GPU): at most 32, also
on images of several megapixels.  The image is 32 and more rows of equal terms d = 1/2 + 2^-20: the
sums k d are exact up to k = 32, and beyond, where 2^-20 is half an ulp of them, every addition
loses it, which makes 16 * 2^-24 of a sum of 64 terms.  The tree over the lanes doubles equal
numbers and the workgroups' sums are added in binary64, both exact, so what is left is the rounding
of 1/n, of the sum to binary32 and of their product: 3 * 2^-24."""
import numpy as np
import pytest

from splatrs_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(256, 32), (2048, 2560)])
def test_l1_of_equal_terms(width, height):
    print(f"[gpu-case] L1 of equal terms {width}x{height}", flush=True)
    ctx = abi.Context(0)
    d = np.float32(0.5 + 2.0 ** -20)
    x = np.full((height, width, 3), d, np.float32)
    loss, _ = ctx.photometric_loss(x, np.zeros_like(x), width, height, 0.0)
    ctx.close()
    err = abs(float(loss) / float(d) - 1.0)
    assert err <= 3 * 2.0 ** -24, err * 2 ** 24
