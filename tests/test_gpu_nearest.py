"""Nearest neighbours over boxes of 64 points in Morton order (needs a gfx950 GPU): clouds on
both sides of the brute-force limit, with a last block of one point, more than 64 blocks and
more than 64 blocks of blocks, against the definition: the three smallest (distance, index)
pairs of the other points, grouped where their coordinates have the same bits, in binary64 and
exactly."""
import numpy as np
import pytest

from splatrs_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


def definition(pts, queries):
    out = []
    p = pts.astype(np.float64)
    bits = np.ascontiguousarray(pts).view(np.uint32)
    with np.errstate(invalid="ignore"):
        for i in queries:
            e = p[i] - p
            d = e[:, 0] * e[:, 0] + e[:, 1] * e[:, 1] + e[:, 2] * e[:, 2]
            d[~np.isfinite(d)] = np.inf
            d[i] = np.inf
            cand = np.flatnonzero(d <= np.partition(d, 2)[2])
            order = cand[np.argsort(d[cand], kind="stable")][:3]
            order = [j for j in order if d[j] < np.inf]
            total, k = 0.0, 0
            while k < len(order):
                g = k + 1
                while g < len(order) and np.array_equal(bits[order[g]], bits[order[k]]):
                    g += 1
                total += d[order[k]] * (g - k)
                k = g
            out.append(total / len(order) if len(order) else 0.0)
    return np.array(out)


def cloud(kind, n):
    rng = np.random.default_rng(n)
    pts = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    if kind == "lattice":      # equal distances everywhere
        pts = rng.integers(0, 12, (n, 3)).astype(np.float32) * np.float32(0.25)
    elif kind == "plane":
        pts[:, 1] = 3.0
    elif kind == "same":
        pts[:] = pts[0]
    elif kind == "outliers":   # the rest in few cells; every index order within them
        pts[rng.integers(0, n, 3)] = np.float32([[1e6, 0, 0], [0, -3e7, 5], [2e38, 1, -3e38]])
        pts[n // 2] = pts[n // 3]
    elif kind == "not finite":
        pts[rng.integers(0, n, 40), rng.integers(0, 3, 40)] = np.float32(np.inf)
        pts[rng.integers(0, n, 40), rng.integers(0, 3, 40)] = np.float32(-np.inf)
        pts[rng.integers(0, n, 200), rng.integers(0, 3, 200)] = np.float32(np.nan)
        pts[-70:] = np.float32(np.nan)
        pts[rng.integers(0, n, 40), 0] = np.float32(-0.0)
    return pts


@pytest.mark.parametrize("kind", ["uniform", "lattice", "plane", "same", "outliers",
                                  "not finite"])
@pytest.mark.parametrize("n", [2048, 2049, 4161])
def test_every_point(ctx, kind, n):
    print(f"[gpu-case] {kind} n={n}", flush=True)
    pts = cloud(kind, n)
    assert np.array_equal(ctx.mean_nn_dist2(pts), definition(pts, range(n)))


@pytest.mark.parametrize("kind", ["uniform", "outliers"])
def test_large(ctx, kind):
    n = 64 ** 3 + 4097
    print(f"[gpu-case] {kind} n={n}", flush=True)
    pts = cloud(kind, n)
    q = np.unique(np.concatenate([np.arange(0, n, 2111), [n // 2, n // 3, n - 1]]))
    assert np.array_equal(ctx.mean_nn_dist2(pts)[q], definition(pts, q))
