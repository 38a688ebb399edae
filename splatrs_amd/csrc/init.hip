// Initialisation from a point cloud (Model::from_points, src/model.rs:77-104) with the
// mean squared distance to the three nearest other points (mean_nn_dist2,
// src/model.rs:128-186) computed on the GPU.
//
// Distances in binary64.  Small clouds by brute force: each lane owns one query point and
// streams every point through LDS, keeping the three nearest other points.  Larger ones over
// blocks of 64 points in Morton order with bounding boxes: a wave takes the queries of one block
// and visits the blocks whose boxes are near enough.  Both keep the three smallest (distance,
// index) pairs.  The reference queries a kd-tree over the unique positions and walks them by
// distance adding `distance * take`; here candidates at the same position are grouped the same
// way, so the result is the reference's value.
#include <cmath>
#include <cstring>
#include <utility>

#include "internal.hpp"

namespace splat {
namespace {

constexpr int kKnnBlock = 256;

// The mean over the (up to) three nearest other points j0, j1, j2 at the squared distances
// d0 <= d1 <= d2 (index 0xffffffff: none).
__device__ __forceinline__ double mean_of_nearest(const float* __restrict__ xyz, double d0,
                                                  double d1, double d2, uint32_t j0, uint32_t j1,
                                                  uint32_t j2) {
  // Walk the candidates by distance, grouping points at the same position.
  const double ds[3] = {d0, d1, d2};
  const uint32_t js[3] = {j0, j1, j2};
  double sum = 0.0;
  uint32_t counted = 0;
  for (int c = 0; c < 3;) {
    if (js[c] == 0xffffffffu) break;
    const uint32_t a = js[c];
    int g = c + 1;
    // same position = the same bits in all three coordinates (the reference's key)
    while (g < 3 && js[g] != 0xffffffffu &&
           f2bits(xyz[3 * (size_t)js[g]]) == f2bits(xyz[3 * (size_t)a]) &&
           f2bits(xyz[3 * (size_t)js[g] + 1]) == f2bits(xyz[3 * (size_t)a + 1]) &&
           f2bits(xyz[3 * (size_t)js[g] + 2]) == f2bits(xyz[3 * (size_t)a + 2]))
      g++;
    const uint32_t take = (uint32_t)(g - c);
    sum += ds[c] * (double)take;
    counted += take;
    c = g;
  }
  return counted > 0 ? sum / (double)counted : 0.0;
}

__global__ void __launch_bounds__(kKnnBlock) knn3_kernel(const float* __restrict__ xyz, uint32_t n,
                                                         double* __restrict__ out) {
  __shared__ double sp[kKnnBlock * 3];
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < n;
  const double qx = valid ? (double)xyz[3 * (size_t)i] : 0.0;
  const double qy = valid ? (double)xyz[3 * (size_t)i + 1] : 0.0;
  const double qz = valid ? (double)xyz[3 * (size_t)i + 2] : 0.0;
  double d0 = INFINITY, d1 = INFINITY, d2 = INFINITY;
  uint32_t j0 = 0xffffffffu, j1 = 0xffffffffu, j2 = 0xffffffffu;
  for (uint32_t base = 0; base < n; base += kKnnBlock) {
    __syncthreads();
    const uint32_t jl = base + threadIdx.x;
    if (jl < n) {
      sp[3 * threadIdx.x] = (double)xyz[3 * (size_t)jl];
      sp[3 * threadIdx.x + 1] = (double)xyz[3 * (size_t)jl + 1];
      sp[3 * threadIdx.x + 2] = (double)xyz[3 * (size_t)jl + 2];
    }
    __syncthreads();
    const uint32_t cnt = min((uint32_t)kKnnBlock, n - base);
    for (uint32_t k = 0; k < cnt; k++) {
      const uint32_t j = base + k;
      const double dx = qx - sp[3 * k], dy = qy - sp[3 * k + 1], dz = qz - sp[3 * k + 2];
      const double d = dx * dx + dy * dy + dz * dz;  // SquaredEuclidean, x, y, z in order
      if (j == i || !(d < d2)) continue;
      if (d < d1) {
        d2 = d1;
        j2 = j1;
        if (d < d0) {
          d1 = d0;
          j1 = j0;
          d0 = d;
          j0 = j;
        } else {
          d1 = d;
          j1 = j;
        }
      } else {
        d2 = d;
        j2 = j;
      }
    }
  }
  if (valid) out[i] = mean_of_nearest(xyz, d0, d1, d2, j0, j1, j2);
}

// ---- larger clouds ----------------------------------------------------------------------

constexpr uint32_t kKnnHalf = 8;  // Morton bits per axis and sort: two sorts, 16 bits per axis
constexpr size_t kKnnBruteMax = 2560;  // see mean_nn_dist2_dev

constexpr uint32_t kKnnQueries = 16;

// The three smallest (distance, index) pairs: what a walk of all points in index order keeps.
struct Nearest3 {
  double d0 = INFINITY, d1 = INFINITY, d2 = INFINITY;
  uint32_t j0 = 0xffffffffu, j1 = 0xffffffffu, j2 = 0xffffffffu;
  __device__ __forceinline__ void add(double d, uint32_t j) {
    if (!(d < d2 || (d == d2 && j < j2))) return;
    const bool b1 = d < d1 || (d == d1 && j < j1), b0 = d < d0 || (d == d0 && j < j0);
    d2 = b1 ? d1 : d;
    j2 = b1 ? j1 : j;
    d1 = b0 ? d0 : b1 ? d : d1;
    j1 = b0 ? j0 : b1 ? j : j1;
    d0 = b0 ? d : d0;
    j0 = b0 ? j : j0;
  }
};

__device__ __forceinline__ float lane_value(float v, uint32_t lane) {
  return bits2f((uint32_t)__builtin_amdgcn_readlane((int)f2bits(v), (int)lane));
}

__device__ __forceinline__ bool finite3(float x, float y, float z) {
  return fabsf(x) < INFINITY && fabsf(y) < INFINITY && fabsf(z) < INFINITY;
}
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fminf(v, __shfl_xor(v, d, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
  return v;
}

// bounds[0..2] / [3..5]: the range of most coordinates, from 256 points spread over the cloud:
// all but the 4 least and the 4 greatest of an axis' finite ones.  (The least and greatest of
// all points would put a scene into one cell if a single point lies far outside it.)
constexpr uint32_t kKnnSamples = 256, kKnnTail = 4;
__global__ void __launch_bounds__(kKnnSamples) knn_bounds_kernel(const float* __restrict__ xyz,
                                                                 uint32_t n,
                                                                 float* __restrict__ bounds) {
  __shared__ float s[3][kKnnSamples];
  const uint32_t k = threadIdx.x;
  const size_t i = (size_t)((uint64_t)k * n / kKnnSamples);
  const float p[3] = {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]};
  const bool finite = finite3(p[0], p[1], p[2]);
#pragma unroll
  for (int c = 0; c < 3; c++) s[c][k] = finite ? p[c] : INFINITY;
  const uint32_t count = (uint32_t)__syncthreads_count(finite ? 1 : 0);
  const uint32_t tail = min(kKnnTail, count / 4);
  if (k < 6 && count == 0) bounds[k] = 0.0f;
  uint32_t rank[3] = {0, 0, 0};
  for (uint32_t j = 0; j < kKnnSamples; j++)
#pragma unroll
    for (int c = 0; c < 3; c++)
      rank[c] += s[c][j] < p[c] || (s[c][j] == p[c] && j < k) ? 1u : 0u;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    if (finite && rank[c] == tail) bounds[c] = p[c];
    if (finite && rank[c] == count - 1 - tail) bounds[3 + c] = p[c];
  }
}

// Bits 0..7 of x to bits 0, 3, 6, ...
__device__ __forceinline__ uint32_t spread3(uint32_t x) {
  x = (x | (x << 8)) & 0x0000f00fu;
  x = (x | (x << 4)) & 0x000c30c3u;
  return (x | (x << 2)) & 0x00249249u;
}

// Item k's half of the Morton code: of point k (`order` null, the lower half, first sort) or of
// point order[k] (the upper half; points that are not finite behind all others).  16 bits per
// axis keep the cells of a scene small next to points far outside it.
__global__ void __launch_bounds__(256) knn_keys_kernel(const float* __restrict__ xyz, uint32_t n,
                                                       const float* __restrict__ bounds,
                                                       const uint32_t* __restrict__ order,
                                                       uint32_t* __restrict__ keys,
                                                       uint32_t* __restrict__ vals) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t i = order ? order[k] : k;
  const float p[3] = {xyz[3 * (size_t)i], xyz[3 * (size_t)i + 1], xyz[3 * (size_t)i + 2]};
  uint32_t code = 1u << (3 * kKnnHalf);
  if (finite3(p[0], p[1], p[2])) {
    code = 0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      // any monotone cell will do: the boxes are taken from the points.  The cells cover the
      // bounds and a quarter of their span on either side; points beyond share the last cells.
      const double lo = bounds[c], span = (double)bounds[3 + c] - lo;
      const double at = span > 0 ? ((double)p[c] - lo) / span + 0.25 : 0.0;
      const double top = (double)((1u << 2 * kKnnHalf) - 1u);
      const uint32_t cell = (uint32_t)fmin(fmax(at * (1.0 / 1.5) * (top + 1.0), 0.0), top);
      code |= spread3(order ? cell >> kKnnHalf : cell & ((1u << kKnnHalf) - 1u)) << c;
    }
  }
  keys[k] = code;
  if (!order) vals[k] = k;
}

// A block's 64 points in Morton order, {x, y, z, index}, their box (of the finite ones) and, as
// bits in lo.w, their least index.
__global__ void __launch_bounds__(64) knn_blocks_kernel(const float* __restrict__ xyz, uint32_t n,
                                                        const uint32_t* __restrict__ order,
                                                        float4* __restrict__ pts,
                                                        float4* __restrict__ lo,
                                                        float4* __restrict__ hi) {
  const uint32_t q = blockIdx.x * 64 + threadIdx.x;
  float4 a = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
  float4 b = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
  if (q < n) {
    const uint32_t i = order[q];
    const float x = xyz[3 * (size_t)i], y = xyz[3 * (size_t)i + 1], z = xyz[3 * (size_t)i + 2];
    pts[q] = make_float4(x, y, z, bits2f(i));
    if (finite3(x, y, z)) a = b = make_float4(x, y, z, 0.0f);
  }
  uint32_t least = q < n ? order[q] : 0xffffffffu;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) least = min(least, (uint32_t)__shfl_xor((int)least, d, 64));
  a = make_float4(wave_min(a.x), wave_min(a.y), wave_min(a.z), bits2f(least));
  b = make_float4(wave_max(b.x), wave_max(b.y), wave_max(b.z), 0.0f);
  if (threadIdx.x == 0) {
    lo[blockIdx.x] = a;
    hi[blockIdx.x] = b;
  }
}

// The boxes of 64 consecutive blocks each.
__global__ void __launch_bounds__(64) knn_supers_kernel(uint32_t nb, const float4* __restrict__ lo,
                                                        const float4* __restrict__ hi,
                                                        float4* __restrict__ slo,
                                                        float4* __restrict__ shi) {
  const uint32_t q = min(blockIdx.x * 64 + threadIdx.x, nb - 1);  // repeating one changes nothing
  const float4 a = lo[q], b = hi[q];
  const float4 c = make_float4(wave_min(a.x), wave_min(a.y), wave_min(a.z), 0.0f);
  const float4 d = make_float4(wave_max(b.x), wave_max(b.y), wave_max(b.z), 0.0f);
  if (threadIdx.x == 0) {
    slo[blockIdx.x] = c;
    shi[blockIdx.x] = d;
  }
}

// Squared distance between boxes [alo, ahi] and [blo, bhi], rounded as the distance of two
// points is: each gap is the rounded difference of coordinates at least as close as those of
// any two points of the boxes, and rounding is monotone, so it is never above their distance
// and a block is left out only if none of its points could enter a query's three.
__device__ __forceinline__ double box_dist2(float4 alo, float4 ahi, float4 blo, float4 bhi) {
  const double dx = fmax(fmax((double)blo.x - (double)ahi.x, (double)alo.x - (double)bhi.x), 0.0);
  const double dy = fmax(fmax((double)blo.y - (double)ahi.y, (double)alo.y - (double)bhi.y), 0.0);
  const double dz = fmax(fmax((double)blo.z - (double)ahi.z, (double)alo.z - (double)bhi.z), 0.0);
  return dx * dx + dy * dy + dz * dz;
}

// Sixteen consecutive queries in Morton order per wave, four lanes each: lane 16 s + q looks at
// every fourth point of a block, from the s-th, for query q.  First the queries' own and the
// neighbouring blocks, for a bound, then every block whose box may hold a closer point (64 boxes
// of blocks of blocks, then of blocks, tested at a time, one per lane, against the box of the
// queries and the largest of their bounds; then by each query); at the end the four lanes' lists
// are merged.  A candidate's distance is first taken in binary32, with room for its rounding, and
// in binary64 only where that leaves it possible.  Bound by the latency of a block visit (points
// loaded while the previous block is looked at): 294 us for 150k points
// on twenty ellipsoids with 2 % in a box of six times their size (381 us with cells over all
// points' range; a lane per query and 64 queries per wave, all distances in binary64, took three
// times as long, its last waves those of the points far out).
__global__ void __launch_bounds__(64) knn_query_kernel(const float* __restrict__ xyz, uint32_t n,
                                                       uint32_t nb, uint32_t ns,
                                                       const float4* __restrict__ pts,
                                                       const float4* __restrict__ lo,
                                                       const float4* __restrict__ hi,
                                                       const float4* __restrict__ slo,
                                                       const float4* __restrict__ shi,
                                                       double* __restrict__ out) {
  __shared__ float4 sp[64];
  const uint32_t lane = threadIdx.x, slice = lane >> 4;
  const uint32_t q = blockIdx.x * kKnnQueries + (lane & 15u), own = blockIdx.x / 4;
  const float4 me = q < n ? pts[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const uint32_t i = f2bits(me.w);
  const bool valid = q < n && finite3(me.x, me.y, me.z);  // others have no near point
  const double qx = me.x, qy = me.y, qz = me.z;
  Nearest3 best;
  if (!valid) best.d2 = -1.0;
  // d2 with room for the rounding of a binary32 distance: relative 2^-21 and, where it
  // underflows, less than 1e-37
  float most32 = valid ? INFINITY : -1.0f;
  const auto load = [&](uint32_t b) {  // uniform b
    const uint32_t k = b * 64 + lane;
    return k < n ? pts[k] : make_float4(NAN, NAN, NAN, 0.0f);
  };
  const auto visit = [&](float4 p) {
    __syncthreads();  // the previous block's points are no longer read
    sp[lane] = p;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < 64; k += 4) {
      const float4 c = sp[k + slice];
      const float ex = me.x - c.x, ey = me.y - c.y, ez = me.z - c.z;
      if (!(ex * ex + ey * ey + ez * ez <= most32)) continue;  // also NaN
      const double dx = qx - c.x, dy = qy - c.y, dz = qz - c.z;
      const double d = dx * dx + dy * dy + dz * dz;  // SquaredEuclidean, x, y, z in order
      const uint32_t j = f2bits(c.w);
      if (j == i || !(d < INFINITY)) continue;
      best.add(d, j);
      most32 = fminf(most32, (float)(best.d2 * 1.000001) + 1e-37f);
    }
  };
  // the least third distance of a query's lanes, and the largest of those over the queries
  double mine, most;
  const auto bounds = [&] {
    mine = fmin(best.d2, __shfl_xor(best.d2, 16, 64));
    mine = fmin(mine, __shfl_xor(mine, 32, 64));
    most = mine;
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) most = fmax(most, __shfl_xor(most, d, 64));
    if (valid) most32 = (float)(mine * 1.000001) + 1e-37f;
  };
  // Of the boxes in `mask` (one per lane), those near enough to a query: a box at a time costs
  // more than a query at a time where many are left (queries far apart: a point outside the
  // scene beside points of it).
  const auto refine = [&](uint64_t mask, float4 blo, float4 bhi) {
    if (__popcll(mask) <= (int)kKnnQueries) return mask;
    uint64_t keep = 0;
    for (uint32_t k = 0; k < kKnnQueries; k++) {
      const float4 at = make_float4(lane_value(me.x, k), lane_value(me.y, k),
                                    lane_value(me.z, k), 0.0f);
      keep |= __ballot(box_dist2(at, at, blo, bhi) <= __shfl(mine, (int)k, 64));
    }
    return mask & keep;
  };
  if (__any(valid)) {
    constexpr uint32_t kNear = 2;
    const uint32_t first = own > kNear ? own - kNear : 0u, last = min(own + kNear, nb - 1);
    float4 p = load(own);
    for (uint32_t b = first; b <= last; b++) {  // own, then the others in order
      const uint32_t next = b < own ? b : b + 1;
      const float4 pn = load(min(next, last));
      visit(p);
      p = pn;
    }
    bounds();
    const float4 plo = make_float4(me.x, me.y, me.z, 0.0f);
    const float4 wlo = make_float4(wave_min(valid ? me.x : INFINITY),
                                   wave_min(valid ? me.y : INFINITY),
                                   wave_min(valid ? me.z : INFINITY), 0.0f);
    const float4 whi = make_float4(wave_max(valid ? me.x : -INFINITY),
                                   wave_max(valid ? me.y : -INFINITY),
                                   wave_max(valid ? me.z : -INFINITY), 0.0f);
    for (uint32_t s0 = 0; s0 < ns; s0 += 64) {
      const uint32_t sk = min(s0 + lane, ns - 1);
      const float4 alo = slo[sk], ahi = shi[sk];
      uint64_t supers = refine(
          __ballot(s0 + lane < ns && box_dist2(wlo, whi, alo, ahi) <= most), alo, ahi);
      while (supers) {
        const uint32_t base = (s0 + (uint32_t)__builtin_ctzll(supers)) * 64;
        supers &= supers - 1;
        const uint32_t bk = base + lane;
        const float4 blo = lo[min(bk, nb - 1)], bhi = hi[min(bk, nb - 1)];
        const double bd = box_dist2(wlo, whi, blo, bhi);
        uint64_t blocks = refine(
            __ballot(bk < nb && (bk < first || bk > last) && bd <= most), blo, bhi);
        if (!blocks) continue;
        uint32_t k = (uint32_t)__builtin_ctzll(blocks);
        float4 p = load(base + k);
        while (true) {
          blocks &= blocks - 1;
          const uint32_t kn = blocks ? (uint32_t)__builtin_ctzll(blocks) : k;
          const float4 pn = load(base + kn);
          const float4 clo = make_float4(lane_value(blo.x, k), lane_value(blo.y, k),
                                         lane_value(blo.z, k), lane_value(blo.w, k));
          const float4 chi = make_float4(lane_value(bhi.x, k), lane_value(bhi.y, k),
                                         lane_value(bhi.z, k), 0.0f);
          const double d = box_dist2(plo, plo, clo, chi);
          if (__any(valid && (d < mine || (d == mine && d == best.d2 &&
                                           f2bits(clo.w) < best.j2)))) {
            visit(p);
            bounds();
            blocks &= __ballot(bd <= most);
          }
          if (!blocks) break;
          if (!(blocks >> kn & 1ull)) {  // that one fell out
            k = (uint32_t)__builtin_ctzll(blocks);
            p = load(base + k);
          } else {
            k = kn;
            p = pn;
          }
        }
      }
    }
  }
#pragma unroll
  for (int x = 16; x <= 32; x *= 2) {
    const double e0 = __shfl_xor(best.d0, x, 64), e1 = __shfl_xor(best.d1, x, 64),
                 e2 = __shfl_xor(best.d2, x, 64);
    const uint32_t k0 = (uint32_t)__shfl_xor((int)best.j0, x, 64),
                   k1 = (uint32_t)__shfl_xor((int)best.j1, x, 64),
                   k2 = (uint32_t)__shfl_xor((int)best.j2, x, 64);
    best.add(e0, k0);
    best.add(e1, k1);
    best.add(e2, k2);
  }
  if (q < n && slice == 0)
    out[i] = valid ? mean_of_nearest(xyz, best.d0, best.d1, best.d2, best.j0, best.j1, best.j2)
                   : 0.0;
}

}  // namespace

// Brute force costs a chain of n distances per lane, 90 us per 1000 points, and n^2 once the chip
// is full; the boxes cost 21 small launches (the Morton order is 140 us of them) and then about
// n log n.  A whole call in us, brute force / boxes, points in a cube: 2049 246 / 267, 2500
// 291 / 281, 3000 336 / 303, 5000 521 / 364, 16000 1402 / 357, 50000 4165 / 412, 150000
// 14090 / 645; all points the same: 2500 251 / 252, 150000 13944 / 3071; on a shell with 2 % up to
// twenty radii out: 150000 14136 / 880; in a cube with one point 10^7 away: 150000 14130 / 628
// (cells over all points' range: 14127).
void mean_nn_dist2_dev(splat_ctx* ctx, const float* xyz, size_t n, double* out) {
  if (n <= kKnnBruteMax) {
    launch(ctx, "knn3", knn3_kernel, dim3(blocks_for(n, kKnnBlock)), dim3(kKnnBlock), 0, xyz,
           (uint32_t)n, out);
    return;
  }
  SPLAT_REQUIRE(n < 0xffffffffull - 64, "too many points");
  const unsigned nb = blocks_for(n, 64), ns = blocks_for(nb, 64);
  float* bounds = ctx->buf<float>("knn_bounds", 6);
  uint32_t* k0 = ctx->buf<uint32_t>("knn_k0", n);
  uint32_t* v0 = ctx->buf<uint32_t>("knn_v0", n);
  uint32_t* k1 = ctx->buf<uint32_t>("knn_k1", n);
  uint32_t* v1 = ctx->buf<uint32_t>("knn_v1", n);
  uint32_t* counts = ctx->buf<uint32_t>("knn_counts", radix_count_words(n));
  uint32_t* sums =
      ctx->buf<uint32_t>("knn_sums", scan_temp_bytes(radix_count_words(n)) / sizeof(uint32_t));
  float4* pts = ctx->buf<float4>("knn_pts", n);
  float4* boxes = ctx->buf<float4>("knn_boxes", 2 * (size_t)nb + 2 * (size_t)ns);
  float4 *lo = boxes, *hi = lo + nb, *slo = hi + nb, *shi = slo + ns;
  launch(ctx, "knn_bounds", knn_bounds_kernel, dim3(1), dim3(kKnnSamples), 0, xyz, (uint32_t)n,
         bounds);
  launch(ctx, "knn_keys", knn_keys_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, xyz,
         (uint32_t)n, (const float*)bounds, (const uint32_t*)nullptr, k0, v0);
  if (radix_sort_pairs(ctx, k0, v0, k1, v1, n, (uint32_t)n, nullptr, 3 * kKnnHalf, counts, sums,
                       nullptr)) {
    std::swap(k0, k1);
    std::swap(v0, v1);
  }
  launch(ctx, "knn_keys", knn_keys_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, xyz,
         (uint32_t)n, (const float*)bounds, (const uint32_t*)v0, k0, (uint32_t*)nullptr);
  const int c = radix_sort_pairs(ctx, k0, v0, k1, v1, n, (uint32_t)n, nullptr, 3 * kKnnHalf + 1,
                                 counts, sums, nullptr);
  launch(ctx, "knn_blocks", knn_blocks_kernel, dim3(nb), dim3(64), 0, xyz, (uint32_t)n,
         (const uint32_t*)(c ? v1 : v0), pts, lo, hi);
  launch(ctx, "knn_supers", knn_supers_kernel, dim3(ns), dim3(64), 0, nb, (const float4*)lo,
         (const float4*)hi, slo, shi);
  launch(ctx, "knn_query", knn_query_kernel, dim3(blocks_for(n, kKnnQueries)), dim3(64), 0, xyz, (uint32_t)n, nb, ns,
         (const float4*)pts, (const float4*)lo, (const float4*)hi, (const float4*)slo,
         (const float4*)shi, out);
}

}  // namespace splat

using namespace splat;

extern "C" {

int splat_mean_nn_dist2(splat_ctx* ctx, const float* xyz, uint64_t n, double* out) {
  if (!ctx) return SPLAT_ERR_INVALID;
  try {
    SPLAT_HIP(hipSetDevice(ctx->device));
    SPLAT_REQUIRE(n == 0 || (xyz && out), "null argument");
    if (n < 2) {
      for (uint64_t i = 0; i < n; i++) out[i] = 0.0;
      return SPLAT_OK;
    }
    float* dx = ctx->buf<float>("knn_xyz", 3 * n);
    double* dd = ctx->buf<double>("knn_out", n);
    SPLAT_HIP(hipMemcpyAsync(dx, xyz, 3 * n * 4, hipMemcpyHostToDevice, ctx->stream));
    mean_nn_dist2_dev(ctx, dx, n, dd);
    SPLAT_HIP(hipMemcpyAsync(out, dd, n * 8, hipMemcpyDeviceToHost, ctx->stream));
    SPLAT_HIP(hipStreamSynchronize(ctx->stream));
    ctx->err.clear();
    return SPLAT_OK;
  } catch (const Error& e) {
    ctx->err = e.msg;
    return e.code;
  }
}

int splat_from_points(splat_ctx* ctx, const float* xyz, const uint8_t* rgb, uint64_t n,
                      float* gaussians) {
  if (!ctx) return SPLAT_ERR_INVALID;
  if (n && (!xyz || !rgb || !gaussians)) {
    ctx->err = "null argument";
    return SPLAT_ERR_INVALID;
  }
  std::vector<double> d2(n);
  const int st = splat_mean_nn_dist2(ctx, xyz, n, d2.data());
  if (st != SPLAT_OK) return st;
  const float opacity = logf(0.1f / (1.0f - 0.1f));  // inverse_sigmoid(0.1), math.rs:395-397
  const float sh_c0 = (float)0.28209479177387814;
  for (uint64_t i = 0; i < n; i++) {
    float* g = gaussians + i * kParams;
    std::memset(g, 0, kParams * sizeof(float));
    const float dd = rmax((float)d2[i], 1e-7f);
    const float log_s = logf(sqrtf(dd));
    for (int c = 0; c < 3; c++) {
      g[c] = xyz[3 * i + c];
      g[3 + c] = log_s;
      g[11 + c] = ((float)rgb[3 * i + c] / 255.0f - 0.5f) / sh_c0;  // rgb_to_sh, sh.rs:41-43
    }
    g[6] = 1.0f;
    g[10] = opacity;
  }
  return SPLAT_OK;
}

}  // extern "C"
