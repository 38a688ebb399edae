"""Models on their way to host memory (needs a gfx950 GPU): chunks of 4096 records through a ring
of 12, one thread and several, one array and three; what was restored comes back bit for bit, also
into memory downloaded to before and from two trainers of one context in turn."""
import numpy as np
import pytest

from splatrs_amd import abi
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 12 * 4096, 12 * 4096 + 1, 150_001])
def test_comes_back(ctx, n):
    print(f"[gpu-case] download n={n}", flush=True)
    rng = np.random.default_rng(n)
    words = lambda: rng.integers(0, 1 << 30, (n, rec.NUM_PARAMS), dtype=np.uint32).view(np.float32)
    a, b = abi.Trainer(ctx, words()), abi.Trainer(ctx, words())
    for _ in range(2):
        states = [dict(params=words(), m=words(), v=words()) for _ in range(2)]
        for t, s in zip((a, b), states):
            t.restore(s, 3)
        for t, s in zip((a, b), states):
            one, all3 = t.download(), t.download(moments=True)
            assert np.array_equal(one["params"].view(np.uint32), s["params"].view(np.uint32))
            for key in s:
                assert np.array_equal(all3[key].view(np.uint32), s[key].view(np.uint32)), key
    a.close()
    b.close()
