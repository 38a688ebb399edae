"""A model downloaded to device memory (needs a gfx950 GPU): where the caller's array is on the
device, the records go there by the runtime's own copy, which checks the range; they are those of
a download to the host, and what lies behind the array stays."""
import ctypes as C

import numpy as np
import pytest
import torch

from splatrs_amd import abi
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4097])
def test_to_device_memory(n):
    print(f"[gpu-case] download of {n} rows to device memory", flush=True)
    ctx = abi.Context(0)
    rng = np.random.default_rng(n)
    words = lambda: rng.integers(0, 1 << 30, (n, rec.NUM_PARAMS), dtype=np.uint32).view(np.float32)
    t = abi.Trainer(ctx, words())
    t.restore(dict(params=words(), m=words(), v=words()), 3)
    want = t.download(moments=True)
    out = torch.full((3, n * rec.NUM_PARAMS + 64), 7.0, device="cuda")
    torch.cuda.synchronize()
    at = [C.c_void_p(out[k].data_ptr()) for k in range(3)]
    ctx.check(abi.lib().splat_trainer_download(t._h, at[0], at[1], at[2], None, None, None, n),
              "trainer_download")
    got = out.cpu().numpy()
    t.close()
    ctx.close()
    for k, name in enumerate(("params", "m", "v")):
        rows = got[k, :-64].reshape(n, rec.NUM_PARAMS)
        assert np.array_equal(rows.view(np.uint32), want[name].view(np.uint32)), name
        assert (got[k, -64:] == 7.0).all()
