"""Tiles beyond the 4096 entries that are sorted in LDS, and many queued tiles at once (needs a
gfx950 GPU).  Chunks of 4096 are merged pair by pair: one chunk over, a pair with a last run of
one entry, odd numbers of chunks over several rounds, and more segments than splits are held
(512).  The lists are whole numbers and equal the oracle's exactly.  The time of a tile grows
with n log n: eight times the entries take well below the 64 times of a quadratic sort."""
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


def rows(rng, n):
    p = np.zeros(n, rec.PROJ)
    p["radius"], p["opacity"] = 1, 0.5
    p["conic"] = [0.1, 0.0, 0.1]
    p["depth"] = rng.choice(rng.uniform(0.3, 9.0, max(2, n // 3)), n).astype(np.float32)
    p["tile_max"] = [1, 1]
    return p


def check(ctx, p, width):
    g, o = ctx.bin(p, width, 16), O.bin(p, width, 16)
    assert g.num_entries == o.num_entries
    assert np.array_equal(g.sorted_keys, o.sorted_keys)
    assert np.array_equal(g.sorted_entries, o.sorted_entries)
    assert np.array_equal(g.tile_range, o.tile_range)


@pytest.mark.parametrize("n", [4097, 8192, 8193, 12288, 12289, 36865, 2_200_000])
def test_merged_tile(ctx, n):
    print(f"[gpu-case] a tile of {n} entries", flush=True)
    rng = np.random.default_rng(n)
    p = rows(rng, n + 40)
    # behind a tile of 40 entries, so that its lists start at an odd place
    where = rng.permutation(n + 40)[:n]
    p["tile_min"][where], p["tile_max"][where] = [1, 0], [2, 1]
    check(ctx, p, 48)


@pytest.mark.parametrize("kind", ["already sorted", "reversed", "all equal"])
def test_merged_tile_in_order(ctx, kind):
    print(f"[gpu-case] a tile of 20000 entries, {kind}", flush=True)
    p = rows(np.random.default_rng(1), 20000)
    d = np.sort(p["depth"])
    p["depth"] = {"already sorted": d, "reversed": d[::-1], "all equal": d * 0 + 1}[kind]
    check(ctx, p, 16)


def test_many_queued_tiles(ctx):
    """More queued tiles than workgroups (1024), from both ends of the queue, among tiles that
    one wave sorts."""
    tiles = 1500
    print(f"[gpu-case] {tiles} tiles of mixed sizes", flush=True)
    rng = np.random.default_rng(5)
    sizes = np.tile([600, 1100, 40, 513, 2100], tiles // 5)
    sizes[[7, 700]] = 4500, 9000
    tile = rng.permutation(np.repeat(np.arange(tiles), sizes))
    p = rows(rng, len(tile))
    p["tile_min"][:, 0], p["tile_min"][:, 1] = tile, 0
    p["tile_max"][:, 0], p["tile_max"][:, 1] = tile + 1, 1
    check(ctx, p, 16 * tiles)


def test_time_grows_with_n_log_n(ctx):
    print("[gpu-case] sort times of tiles of 32768 and 262144 entries", flush=True)

    def sort_ms(n):
        p = rows(np.random.default_rng(n), n)
        ctx.bin(p, 16, 16)
        ctx.set_timing(True)
        best = np.inf
        for _ in range(3):
            ctx.reset_timing()
            ctx.bin(p, 16, 16)
            best = min(best, ctx.kernel_times()["bin_sort_queue"][1])
        ctx.set_timing(False)
        return best

    assert sort_ms(262144) < 24 * sort_ms(32768)
