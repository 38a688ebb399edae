"""Launch shapes of the compositing kernels on images with few tiles (needs a gfx950 GPU): a set
shape runs as given and the default one takes kernels of its own there, so the walks' edges (see
test_gpu_walk_lists, which runs the default against the oracle) are compared between the two; a
persistent shape also takes the ordered backward's form for many tiles.  Results are the same bits.
Tuning counts the default as a candidate of its own where it is one, and what it reports can be
set."""
import numpy as np
import pytest

from splatrs_amd import abi
from splatrs_amd import records as rec
from test_gpu_walk_lists import CASES, scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


def shape(fwd, fwd_persistent, bwd, bwd_persistent, rows):
    s = np.zeros((), rec.TUNE_RESULT)
    s["fwd_batch"], s["fwd_persistent"], s["fwd_per_cu"] = fwd, fwd_persistent, 2
    s["bwd_batch"], s["bwd_persistent"], s["bwd_per_cu"] = bwd, bwd_persistent, 2
    s["bwd_row_lists"] = rows
    return s


SHAPES = [shape(0, 0, 0, 0, 1), shape(32, 0, 16, 0, 1), shape(64, 0, 32, 0, 1),
          shape(128, 0, 32, 0, 0), shape(256, 0, 16, 0, 0), shape(64, 1, 32, 1, 1),
          shape(256, 1, 16, 1, 0)]


def trained(ctx, g, cam, rgb, shapes, ordered):
    t = abi.Trainer(ctx, g)
    t.add_view(cam, rgb)
    if shapes is not None:
        t.set_shapes(shapes)
    lr = rec.learning_rates(1e-4)
    for absgrad in (False, True):
        t.step(0, rec.step_params(3, lr, accumulate_stats=True, absgrad=absgrad,
                                  ordered_backward=ordered, background=(0.2, 0.5, 0.1)),
               result=False)
    out = t.download(moments=True, stats=True)
    t.close()
    return out


@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("n,sigma_px,width,height,opacity", CASES)
def test_shapes_at_list_and_batch_edges(ctx, n, sigma_px, width, height, opacity, ordered):
    print(f"[gpu-case] shapes: {n} Gaussians of {sigma_px} px, {width}x{height}, "
          f"ordered={ordered}", flush=True)
    g, cam = scene(n, sigma_px, width, height, opacity)
    rgb = np.random.default_rng(n).integers(0, 256, (height, width, 3), dtype=np.uint8)
    want = trained(ctx, g, cam, rgb, None, ordered)
    for s in SHAPES:
        got = trained(ctx, g, cam, rgb, s, ordered)
        for k in want:
            assert np.array_equal(np.asarray(want[k]).view(np.uint8),
                                  np.asarray(got[k]).view(np.uint8)), (s, k)


@pytest.mark.parametrize("ordered,candidates", [(False, 17 + 17), (True, 17 + 8)])
def test_tuning_with_few_tiles(ctx, ordered, candidates):
    print(f"[gpu-case] tuning on few tiles, ordered={ordered}", flush=True)
    g, cam = scene(*CASES[-1])
    height, width = int(cam["height"]), int(cam["width"])
    t = abi.Trainer(ctx, g)
    t.add_view(cam, np.full((height, width, 3), 100, np.uint8))
    p = rec.step_params(3, rec.learning_rates(1e-4), ordered_backward=ordered)
    r = t.tune(0, p)
    assert r["candidates"] == candidates
    assert 0 < r["fwd_ms"] <= r["default_fwd_ms"] and 0 < r["bwd_ms"] <= r["default_bwd_ms"]
    t.set_shapes(r)
    t.step(0, p, result=False)
    for bad in (shape(48, 0, 32, 0, 1), shape(64, 0, 64, 0, 1), shape(-1, 0, 32, 0, 1)):
        with pytest.raises(abi.SplatError):
            t.set_shapes(bad)
    t.close()
