"""Compositing walks where their lists, batches and staging end (needs a gfx950 GPU).

Tiles with entry counts around the sizes of an entry list (32, 64) and of an LDS batch (256),
Gaussians that cover whole tiles (the ordered backward stages at most 1024 pixel terms at a
time, four full tiles), cover one 4x4 sub-block, or mix, on images whose last tiles are one
pixel wide or high.  Forward and ordered backward against the oracle (the same binary32
operations in the same order: bitwise, up to the rare ulp of ln(255 o)); the tree-reduced
backward against the oracle's sums within 1e-4 of each field's largest value, a hundred times
the rounding of a sum of 256 binary32 terms relative to its largest partial sum.
"""
import numpy as np
import pytest

import oracle_lib as O
from splatrs_amd import abi, scenes
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


def scene(n, sigma_px, width, height, opacity):
    """n Gaussians in front of one camera, of about sigma_px pixels (drawn per Gaussian from
    the list), faint enough that the walk goes deep."""
    rng = np.random.default_rng(1000 + n)
    cam = scenes.look_at(width, height, 100.0, 100.0, (0.0, 0.0, -4.0), (0.0, 0.0, 0.0))
    g = scenes.random_gaussians(rng, n)
    g[:, 0] = rng.uniform(-0.02 * width, 0.02 * width, n)
    g[:, 1] = rng.uniform(-0.02 * height, 0.02 * height, n)
    g[:, 2] = rng.uniform(-0.5, 0.5, n)
    g[:, 3:6] = (np.log(rng.choice(sigma_px, n) * 4.0 / 100.0)[:, None]
                 + rng.normal(0, 0.1, (n, 3)))
    g[:, 10] = rng.normal(opacity, 0.3, n)
    return g.astype(np.float32), cam


CASES = [
    # n, screen sizes in pixels, width, height, mean opacity logit
    (1, [40.0], 16, 16, 0.0),
    (31, [40.0], 17, 16, -3.0),
    (32, [40.0], 16, 17, -3.0),
    (33, [40.0], 33, 1, -3.0),
    (64, [40.0], 16, 16, -4.0),
    (65, [30.0], 1, 49, -4.0),
    (257, [20.0], 31, 15, -4.5),
    (700, [1.0], 47, 33, 0.0),
    (700, [0.5, 1.0, 4.0, 25.0], 65, 63, -2.0),
]


@pytest.mark.parametrize("n,sigma_px,width,height,opacity", CASES)
def test_walks_at_list_and_batch_edges(ctx, n, sigma_px, width, height, opacity):
    print(f"[gpu-case] {n} Gaussians of {sigma_px} px, {width}x{height}", flush=True)
    g, cam = scene(n, sigma_px, width, height, opacity)
    po = O.project_all(g, cam, rec.proj_opts(3))
    bo = O.bin(po, width, height)
    st = rec.raster_settings(width, height, (0.2, 0.5, 0.1))
    ig, tg, ng = ctx.rasterize_forward(po, bo, st)
    io, to, no = O.rasterize_forward(po, bo, st)
    assert np.abs(ig - io).max() <= 1e-5 and np.abs(tg - to).max() <= 1e-5
    assert (ig == io).mean() >= 0.999 and (ng == no).mean() >= 0.999
    dimg = np.random.default_rng(n).standard_normal(io.shape).astype(np.float32)
    go, ao = O.rasterize_backward(po, bo, st, to, no, dimg)
    for ordered in (True, False):
        gg, ag = ctx.rasterize_backward(po, bo, st, to, no, dimg, ordered=ordered)
        a = np.concatenate([gg.view(np.float32).reshape(n, 9), ag], 1).astype(np.float64)
        b = np.concatenate([go.view(np.float32).reshape(n, 9), ao], 1).astype(np.float64)
        if ordered:
            assert (a == b).mean() >= 0.999, (a == b).mean()
        scale = np.maximum(np.abs(b).max(0), 1e-30)
        assert (np.abs(a - b) <= 1e-4 * np.maximum(np.abs(b), scale)).all()
