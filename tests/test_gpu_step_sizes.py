"""Train steps at the model sizes where the step's launches change (needs a gfx950 GPU): one row,
the rows of a workgroup of the backward tail and one more or less, the sizes where its workgroup
(65536 rows) and the entry-offset scan (16384 rows) change.  In the reference's summation order,
so parameters and moments equal the oracle's bit for bit, up to the rare ulp of ln(255 o)."""
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


@pytest.mark.parametrize("n", [1, 63, 64, 65, 16384, 16385, 65536, 65537])
def test_steps_of(ctx, n):
    print(f"[gpu-case] train steps of {n} Gaussians", flush=True)
    rng = np.random.default_rng(n)
    w, h = 113, 87
    cam = scenes.look_at(w, h, 110.0, 110.0, (0.3, 0.2, -4.0), (0.0, 0.0, 0.0))
    g = scenes.random_gaussians(rng, n, log_scale_mu=-3.0 if n < 1000 else -4.3)
    rgb = rng.integers(0, 256, (h, w, 3), dtype=np.uint8)
    lr = rec.learning_rates(1.6e-4)
    t = abi.Trainer(ctx, g)
    t.add_view(cam, rgb)
    ref = O.TrainState(g)
    for _ in range(2):
        t.step(0, rec.step_params(3, lr, accumulate_stats=True, ordered_backward=True),
               result=False)
        ref.train_step(cam, rgb, 3, lr, accumulate_stats=True)
    got = t.download(moments=True, stats=True)
    t.close()
    for name, want in (("params", ref.params), ("m", ref.m), ("v", ref.v)):
        same = np.mean(got[name].view(np.uint32) == want.view(np.uint32))
        assert same >= 0.999, (name, same)
    assert np.array_equal(got["denom"], ref.denom)
    assert np.array_equal(got["max_radii"], ref.max_radii)
