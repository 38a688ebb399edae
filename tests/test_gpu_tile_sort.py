"""Per-tile sorts at the sizes where they change (needs a gfx950 GPU): one wave up to 512
entries, runs of 128, 256 and 512 ranked in LDS up to 4096, chunks of 4096 beyond, with ties
in depth (broken by the entry index) and a last run or chunk of one entry.  The sorted lists
are whole numbers and equal the oracle's exactly."""
import numpy as np
import pytest

import oracle_lib as O
from splatrs_amd import abi
from splatrs_amd import records as rec

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [511, 512, 513, 769, 1023, 1024, 1025, 2047, 2048, 2049, 3000, 4096, 4097,
                               8193, 20001])
def test_tile_of(ctx, n):
    print(f"[gpu-case] a tile of {n} entries", flush=True)
    rng = np.random.default_rng(n)
    p = np.zeros(n + 70, rec.PROJ)
    p["radius"], p["opacity"] = 1, 0.5
    p["conic"] = [0.1, 0.0, 0.1]
    p["depth"] = rng.choice(rng.uniform(0.3, 9.0, max(2, n // 3)), n + 70).astype(np.float32)
    # n in the second tile of a row of three, the rest spread over the other two and a culled few
    where = rng.permutation(n + 70)
    p["tile_min"][where[:n]] = [1, 0]
    p["tile_max"][where[:n]] = [2, 1]
    p["tile_min"][where[n:n + 30]] = [0, 0]
    p["tile_max"][where[n:n + 30]] = [1, 1]
    p["tile_min"][where[n + 30:n + 60]] = [2, 0]
    p["tile_max"][where[n + 30:n + 60]] = [3, 1]
    p["radius"][where[n + 60:]] = 0
    g, o = ctx.bin(p, 48, 16), O.bin(p, 48, 16)
    assert g.num_entries == o.num_entries == n + 60
    assert np.array_equal(g.sorted_keys, o.sorted_keys)
    assert np.array_equal(g.sorted_entries, o.sorted_entries)
    assert np.array_equal(g.tile_range, o.tile_range)
