"""An image gradient that is not finite at one pixel reaches only the Gaussians that are evaluated
near it (needs a gfx950 GPU): an entry whose rectangle covers a tile, but whose ellipse no pixel of
it lies in, keeps the finite gradient of the pixels it has."""
import numpy as np
import pytest

import oracle_lib as O
from splatrs_amd import abi
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_entry_without_pixels_stays_finite(value, ordered):
    print(f"[gpu-case] dL/dimage {value}, ordered={ordered}", flush=True)
    p = np.zeros(2, rec.PROJ)
    p["mean2d"], p["radius"], p["color"] = [24.0, 24.0], 40, [[0.9, 0.2, 0.4], [0.1, 0.7, 0.3]]
    p["tile_max"] = [3, 3]
    # in front: narrow, along the diagonal; behind it: round, over all tiles
    along, across = 1.0 / 12.0 ** 2, 1.0 / 1.2 ** 2
    p["conic"][0] = [(along + across) / 2, (along - across) / 2, (along + across) / 2]
    p["conic"][1] = [1 / 400.0, 0.0, 1 / 400.0]
    p["depth"], p["opacity"] = [1.0, 2.0], [0.6, 0.5]
    b = O.bin(p, 48, 48)
    st = rec.raster_settings(48, 48, (0.1, 0.2, 0.3))
    image, final_t, n_contrib = O.rasterize_forward(p, b, st)
    dimg = np.random.default_rng(3).standard_normal(image.shape).astype(np.float32)
    want = O.rasterize_backward(p, b, st, final_t, n_contrib, dimg)[0][:1].view(np.float32)
    dimg[8, 40, 0] = value  # in the tile at the upper right, far from the diagonal
    ctx = abi.Context(0)
    got = ctx.rasterize_backward(p, b, st, final_t, n_contrib, dimg, ordered=ordered)[0]
    ctx.close()
    got = got.view(np.float32).reshape(2, 9)
    assert not np.isfinite(got[1]).all()
    # 2304 terms: rounding of a binary32 sum relative to the largest field
    assert np.abs(got[0] - want).max() <= 1e-4 * np.abs(want).max()
