// Tile compositing, forward and backward (src/rasterize.rs:231-505).
//
// One 256-lane workgroup per 16x16 tile, one lane per pixel.  The tile's depth-sorted
// entries are staged through LDS in batches (record gather + per-tile pixel rectangle,
// TileGauss::new at src/rasterize.rs:149-182); every lane walks the batch with its own
// compositing state, exactly the per-pixel walk of the reference's entry-outer loops.  Each
// 16-lane row of a wave (a 4x4 pixel block) walks its own list of the entries that reach it.
// The forward pass stops a workgroup when all its pixels are done.
//
// Backward: each entry's 11 per-pixel terms are reduced over the tile's pixels and
// written to the entry's slots (src/rasterize.rs:449-454); a second kernel sums each
// Gaussian's slots in entry order (src/rasterize.rs:480-503).  The ordered kernel sums the
// pixel terms sequentially in row-major order -- the reference's order, so slots and
// gradients are bitwise identical to it; the tree-reduced kernel sums each row's pixels by
// DPP.
#include "internal.hpp"

namespace splat {
namespace {

// Launches of one view with few tiles in the default shape: each wave's own latency bounds them,
// and registers and LDS are free.  The FEW kernels evaluate a step's pair beside the previous
// step's state update, without a branch, and take larger batches (fewer barriers): the forward
// 256 entries instead of 64, the backward 64 (45 KB of LDS: three workgroups per compute unit)
// instead of 32.  In us, FEW / otherwise, on a light scene (0.15 Gaussians per pixel, in a box)
// and a dense one (0.27, on surfaces):
//   tiles    forward                     backward
//    256     43 /  57   127 / 150        103 / 128   252 / 287
//    900     47 /  61   143 / 167        112 / 137   282 / 322
//   1600     50 /  63   169 / 190        116 / 140   324 / 358
//   2000     46 /  56   153 / 171        104 / 123   288 / 321
//   2700     55 /  56   161 / 175        136 / 118   297 / 335
//   4346     91 /  91   184 / 188        248 / 188   495 / 367
//   5400    112 / 112   225 / 218        315 / 233   611 / 425
// The lines lie where neither scene is slower.  (The general forward with 256 entries is between
// the two up to 2000 tiles and below both from 2700 on, 159 at 4346 on the dense scene; tuning
// finds it.)
constexpr unsigned kFewTilesFwd = 4608;
constexpr unsigned kFewTilesBwd = 1536;
constexpr unsigned kFewTilesOrd = 768;  // see raster_bwd_ordered_kernel
constexpr int kOrdBatch = 32;      // entries staged per batch (ordered backward)

struct TileInfo {
  uint32_t gx0, gy0, w, h;
};

__device__ __forceinline__ TileInfo tile_info(uint32_t tile, uint32_t tiles_x, uint32_t W,
                                              uint32_t H) {  // src/rasterize.rs:198-209
  TileInfo t;
  t.gx0 = (tile % tiles_x) * kTile;
  t.gy0 = (tile / tiles_x) * kTile;
  t.w = min(W - t.gx0, (uint32_t)kTile);
  t.h = min(H - t.gy0, (uint32_t)kTile);
  return t;
}

// Geometry of one tile of the (possibly batched) tile space: its pixel rectangle, the
// width of its view and the view's first pixel in the image buffers.
struct TileGeom {
  TileInfo ti;
  uint32_t width;
  size_t pix0;
};

template <bool BATCH>
__device__ __forceinline__ TileGeom tile_geom(uint32_t tile, uint32_t tiles_x, uint32_t W,
                                              uint32_t H, const BatchDev& bd) {
  TileGeom t;
  if (BATCH) {
    const uint32_t v = find_segment(bd.tile_base, bd.npairs, tile);
    t.ti = tile_info(tile - bd.tile_base[v], bd.tiles_x[v], bd.width[v], bd.height[v]);
    t.width = bd.width[v];
    t.pix0 = bd.pix_base[v];
  } else {
    t.ti = tile_info(tile, tiles_x, W, H);
    t.width = W;
    t.pix0 = 0;
  }
  return t;
}

// The workgroup's next tile: its block index, or (persistent launch) the next one handed
// out by a shared counter.  Every lane sees the same tile.
constexpr uint32_t kXcds = 8;  // accelerator complex dies, each with its own L2

// The die the calling wave runs on (hardware register XCC_ID).
__device__ __forceinline__ uint32_t xcc_id() {
  uint32_t x;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
  return x % kXcds;
}

// Persistent launches: die x takes, from its own counter, the tiles of its eighth of
// [0, T) in index order (neighbouring tiles share Gaussian records in that die's L2), then
// whatever the other eighths have left.  Counters only grow, so every range drains and the
// call returns T once all are taken.  Which die a wave reports only moves work between
// dies; every tile is still taken exactly once.
__device__ __forceinline__ uint32_t take_tile(uint32_t* counter, uint32_t T) {
  const uint32_t x = xcc_id();
  for (uint32_t k = 0; k < kXcds; k++) {
    const uint32_t r = (x + k) % kXcds;
    const uint32_t lo = (uint32_t)((uint64_t)T * r / kXcds);
    const uint32_t hi = (uint32_t)((uint64_t)T * (r + 1) / kXcds);
    const uint32_t t = atomicAdd(&counter[r], 1u);
    if (t < hi - lo) return lo + t;
  }
  return T;
}

// With a dispatch order (tiles by decreasing entry count) the t-th tile taken is order[t];
// a tile's results do not depend on when it runs.
template <bool PERSIST>
__device__ __forceinline__ uint32_t next_tile(uint32_t* counter, uint32_t* s_tile,
                                              const uint32_t* __restrict__ order,
                                              uint32_t num_tiles) {
  uint32_t t;
  if (!PERSIST) {
    t = blockIdx.x;
  } else {
    __syncthreads();  // the previous tile's LDS use is over
    if (threadIdx.x == 0) *s_tile = take_tile(counter, num_tiles);
    __syncthreads();
    t = *s_tile;
  }
  return order && t < num_tiles ? order[t] : t;
}

// Tile-local pixel range of one entry (the clip closure of src/rasterize.rs:158-164).
__device__ __forceinline__ void clip_range(float m, float half, uint32_t offset, uint32_t n,
                                           uint32_t* lo_out, uint32_t* hi_out) {
  const float lo = ceilf((m - half) - 0.5f) - (float)offset;
  const float hi = floorf((m + half) - 0.5f) - (float)offset + 1.0f;
  *lo_out = as_u32(rclamp(lo, 0.0f, (float)n));
  *hi_out = as_u32(rclamp(hi, 0.0f, (float)n));
}

// Tile-local pixel rectangle of an entry as two masks: columns in bits 0-15, rows in bits
// 16-31 (0: empty).
__device__ __forceinline__ uint32_t entry_rect(float4 r0, float4 r1, float4 r2, const TileInfo& t) {
  const float hx = r1.w, hy = r2.x;
  if (!(hx >= 0.0f)) return 0u;  // sigma_max <= 0 or det <= 0: empty
  uint32_t x0, x1, y0, y1;  // all <= 16
  clip_range(r0.x, hx, t.gx0, t.w, &x0, &x1);
  clip_range(r0.y, hy, t.gy0, t.h, &y0, &y1);
  if (x0 >= x1 || y0 >= y1) return 0u;
  return ((1u << x1) - (1u << x0)) | (((1u << y1) - (1u << y0)) << 16);
}

// The records as staged in LDS: conic A (r0.z) and C (r1.x) halved.  Scaling by 1/2
// commutes with every rounding of sigma = 0.5 (A dx dx + C dy dy) + B dx dy
// (src/rasterize.rs:235-236) as long as the products stay normal: a nonzero dx or dy is
// at least 2^-25 (an ulp of a coordinate in [0.5, 2^24)), so for conic entries above 2^-76
// (2D covariances below about 10^22 px^2) (A/2) dx dx + (C/2) dy dy is exactly half of
// A dx dx + C dy dy and the walks get the reference's sigma bit for bit with one multiply
// less.  Uses of the full A and C double them back (exact).
__device__ __forceinline__ float4 half_conic0(float4 r0) {
  r0.z *= 0.5f;
  return r0;
}
__device__ __forceinline__ float4 half_conic1(float4 r1) {
  r1.x *= 0.5f;
  return r1;
}

// Pixel of thread t in the 16x16 tile: wave w = t / 64 covers the 8x8 block
// (w % 2, w / 2); its 16-lane row r = l / 16 the 4x4 sub-block (r % 2, r / 2) of that
// block, and lane l the pixel (l % 4, (l / 4) % 4) of the sub-block.  Square blocks let the
// rectangle tests below cull in both directions, and the backward walks a list of entries
// per row (the DPP reductions are per row).
__device__ __forceinline__ void tile_pixel(uint32_t t, uint32_t* i, uint32_t* j) {
  const uint32_t w = t >> 6, r = (t >> 4) & 3u, q = t & 15u;
  *i = (w & 1u) * 8u + (r & 1u) * 4u + (q & 3u);
  *j = (w >> 1) * 8u + (r >> 1) * 4u + (q >> 2);
}

// Pixels of a rectangle in the 4x4 sub-block of row r of wave w, one bit per lane of the row
// (bit 4 j + i of the sub-block's pixel (i, j)).
__device__ __forceinline__ uint32_t row_mask(uint32_t rc, uint32_t w, uint32_t r) {
  const uint32_t x = (rc >> ((w & 1u) * 8u + (r & 1u) * 4u)) & 0xfu;
  const uint32_t y = (rc >> (16u + (w >> 1) * 8u + (r >> 1) * 4u)) & 0xfu;
  const uint32_t rows = (y | (y << 3) | (y << 6) | (y << 9)) & 0x1111u;  // bit j of y to bit 4 j
  return rows * x;
}

// Whether a rectangle has pixels in the 8x8 block of wave w.
__device__ __forceinline__ bool wave_touches(uint32_t rc, uint32_t w) {
  return ((rc >> ((w & 1u) * 8u)) & 0xffu) != 0 && ((rc >> (16u + (w >> 1) * 8u)) & 0xffu) != 0;
}

__device__ __forceinline__ bool in_rect(uint32_t rc, uint32_t i, uint32_t j) {
  return ((rc >> i) & (rc >> (16u + j)) & 1u) != 0;
}

// The record of a Gaussian in registers, on its way to LDS.
struct StagedRecord {
  float4 a, b, c;
};
__device__ __forceinline__ StagedRecord load_record(const float4* __restrict__ rec, uint32_t g) {
  return StagedRecord{rec[4 * (size_t)g], rec[4 * (size_t)g + 1], rec[4 * (size_t)g + 2]};
}

// A row's entry list in LDS holds words {pixel mask of the row's sub-block << 16 | 16 k} for
// batch entry k: the low half is the entry's byte offset in a float4 array.  Zero is no
// entry (an entry in a list has a pixel).
__device__ __forceinline__ float4 at_bytes(const float4* base, uint32_t bytes) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) + bytes);
}

// Pair counters of the counting instantiations (COUNT = true), one 64-bit word each.
// Forward: visits (steps of a wave's walk, one entry of each of its rows' lists), visits in
// which some lane evaluates its Gaussian, evaluated pairs (sigma in [0, sigma_max]: the
// exponential is computed), passing pairs (alpha >= 1/255 on a pixel still compositing) and
// composited pairs.  Backward: visits, active visits, evaluated and passing pairs of the
// reverse walk.
enum PairCounter : int {
  kFwdVisits, kFwdActive, kFwdEvaluated, kFwdPassing, kFwdComposited,
  kBwdVisits, kBwdActive, kBwdEvaluated, kBwdPassing, kNumPairCounters
};

// Adds a wave's counts to the global counters (lane 0; the counts are wave-uniform).
__device__ __forceinline__ void flush_counts(unsigned long long* pairs, int first,
                                             const uint32_t* c, int n) {
  if ((threadIdx.x & 63) == 0)
    for (int q = 0; q < n; q++)
      if (c[q]) atomicAdd(&pairs[first + q], (unsigned long long)c[q]);
}

// One step of the forward walk for one pixel: evaluate() of src/rasterize.rs:231-244 as far as
// the alpha test.
struct FwdPair {
  uint32_t k16;  // byte offset of the entry
  bool in;       // the pixel is in the entry's rectangle and 0 <= sigma <= sigma_max
  float sigma, o, og;
  __device__ __forceinline__ void evaluate(uint32_t word, uint32_t pixel_bit, const float4* s0,
                                           const float4* s1, float px, float py) {
    k16 = word & 0xffffu;
    const float4 a = at_bytes(s0, k16), b = at_bytes(s1, k16);
    const float dx = px - a.x;
    const float dy = py - a.y;
    sigma = (a.z * dx * dx + b.x * dy * dy) + a.w * dx * dy;  // halved A, C
    in = ((word & pixel_bit) != 0) & !((sigma < 0.0f) | (sigma > b.z));
    o = b.y;
  }
  __device__ __forceinline__ void exponent(const uint64_t* tab) {
    og = o * expf_walk_tab(-sigma, tab);  // used where 0 <= sigma <= sigma_max
  }
};

// The forward pass is bound by VALU issue, so it is built for few walk steps and few
// instructions in each: the four 16-lane rows of a wave walk lists of their own (against one
// walk of the entries that reach the wave's 8x8 block: about a fifth fewer steps), and a list
// word carries the pixels of the row's sub-block that the entry's rectangle holds, one AND
// instead of four comparisons.  10k Gaussians, 256x256: 82 -> 63 us; with 256 entries per batch
// and records prefetched too, 1M Gaussians, 1920x1080: 227 -> 190 us.
// B: entries per LDS batch; BATCH: tiles of many views (BatchDev); PERSIST: a fixed grid
// that takes tiles from `counter` until `num_tiles` are done; COUNT: also count pairs
// into `pairs` (PairCounter); FEW: for launches with few tiles (kFewTilesFwd).
template <int B, bool BATCH, bool PERSIST, bool COUNT = false, bool FEW = false>
__global__ void __launch_bounds__(256) raster_fwd_kernel(
    const float4* __restrict__ rec, const uint32_t* __restrict__ tile_start,
    const uint32_t* __restrict__ order,
    const uint32_t* __restrict__ sorted_gauss, uint32_t num_tiles, uint32_t tiles_x, uint32_t W,
    uint32_t H, float bg0, float bg1, float bg2, float* __restrict__ image,
    float* __restrict__ final_t, uint32_t* __restrict__ n_contrib, BatchDev bd,
    uint32_t* __restrict__ counter, unsigned long long* __restrict__ pairs) {
  static_assert(B <= 256, "each of the 256 lanes stages at most one entry of a batch");
  constexpr int kList = B < 64 ? B : 64;  // entries per list: one ballot covers them
  __shared__ uint64_t tab[32];
  __shared__ float4 s0[B], s1[B], s2[B];
  __shared__ uint32_t srect[B];
  __shared__ uint32_t slist[16][kList + 1];  // per (wave, row): its entries, front to back
  __shared__ uint32_t s_tile;
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Table[threadIdx.x];
  if (FEW && threadIdx.x < 16) slist[threadIdx.x][kList] = 0u;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4;
  const uint32_t pixel_bit = 0x10000u << (lane & 15u);
  const uint32_t* my_list = slist[wave * 4 + row];
  for (;;) {
  const uint32_t tile = next_tile<PERSIST>(counter, &s_tile, order, num_tiles);
  if (tile >= num_tiles) break;
  const TileGeom tg = tile_geom<BATCH>(tile, tiles_x, W, H, bd);
  const TileInfo ti = tg.ti;
  uint32_t i, j;
  tile_pixel(threadIdx.x, &i, &j);
  const bool valid = i < ti.w && j < ti.h;
  const float px = (float)(ti.gx0 + i) + 0.5f;
  const float py = (float)(ti.gy0 + j) + 0.5f;
  float T = 1.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
  uint32_t nc = 0;
  bool done = !valid;
  uint32_t pcount[5] = {0, 0, 0, 0, 0};
  const uint32_t start = tile_start[tile], end = tile_start[tile + 1];
  // The records of a batch are loaded while the batch before it is walked, their Gaussians one
  // batch earlier still (lanes past the end repeat its last entry).
  StagedRecord sr{};
  uint32_t next_g = 0;
  if (threadIdx.x < B && start < end) {
    sr = load_record(rec, sorted_gauss[min(start + threadIdx.x, end - 1)]);
    next_g = sorted_gauss[min(start + B + threadIdx.x, end - 1)];
  }
  for (uint32_t b0 = start; b0 < end; b0 += B) {
    if (__syncthreads_and(done ? 1 : 0)) break;
    const uint32_t cnt = min((uint32_t)B, end - b0);
    if (threadIdx.x < B) {
      s0[threadIdx.x] = half_conic0(sr.a);
      s1[threadIdx.x] = half_conic1(sr.b);
      s2[threadIdx.x] = sr.c;
      srect[threadIdx.x] = entry_rect(sr.a, sr.b, sr.c, ti);
    }
    __syncthreads();
    if (threadIdx.x < B && b0 + B < end) {
      sr = load_record(rec, next_g);
      next_g = sorted_gauss[min(b0 + 2 * B + threadIdx.x, end - 1)];
    }
    // Predicated form of the per-pixel walk (src/rasterize.rs:262-290): every decision of
    // evaluate() and the T_MIN test is a lane predicate; only the exp is skipped when no
    // lane of the wave needs it.  The four rows of a wave walk, side by side and each in
    // order, the entries whose pixel rectangle reaches the row's 4x4 sub-block.
    for (uint32_t c0k = 0; c0k < cnt; c0k += kList) {
      if (!__any(!done)) break;  // uniform: this wave's pixels are finished
      const uint32_t kl = c0k + min(lane, (uint32_t)kList - 1u);
      const uint32_t rc = kl < cnt && lane < (uint32_t)kList ? srect[kl] : 0u;
      uint32_t steps = 0;
      // the walk of the previous list is over before this one is written: same wave
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
      for (uint32_t r = 0; r < 4; r++) {
        const uint32_t pm = row_mask(rc, wave, r);
        const uint64_t m = __ballot(pm != 0);
        const uint32_t len = (uint32_t)__popcll(m);
        uint32_t* list = slist[wave * 4 + r];
        if (pm) list[__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] =
            (pm << 16) | (kl << 4);
        if (lane >= len && lane < (uint32_t)kList) list[lane] = 0u;  // past the end: no entry
        steps = max(steps, len);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      uint32_t last = 0xffffffffu;  // byte offset of the last composited entry of this list
      const auto blend = [&](const FwdPair& p, bool pass1, float4 c) {
        const bool pass2 = pass1 & !(p.og < kAlphaMin);
        const float alpha = rmin(p.og, kAlphaMax);
        const float test_t = T * (1.0f - alpha);
        const bool stop = test_t < kTMin;
        done = done | (pass2 & stop);
        const bool comp = pass2 & !stop;
        if (COUNT) {
          pcount[3] += (uint32_t)__popcll(__ballot(pass2));
          pcount[4] += (uint32_t)__popcll(__ballot(comp));
        }
        const float w = alpha * T;
        c0 = comp ? c0 + w * c.y : c0;
        c1 = comp ? c1 + w * c.z : c1;
        c2 = comp ? c2 + w * c.w : c2;
        T = comp ? test_t : T;
        last = comp ? p.k16 : last;
      };
      if (FEW) {
        // the pair of the next step is evaluated beside the blend of this one
        FwdPair p;
        p.evaluate(my_list[0], pixel_bit, s0, s1, px, py);
        p.exponent(tab);
        uint32_t next = my_list[1];
        for (uint32_t t = 0; t < steps; t++) {
          const FwdPair now = p;
          const float4 c = at_bytes(s2, now.k16);
          p.evaluate(next, pixel_bit, s0, s1, px, py);
          p.exponent(tab);
          next = my_list[min(t + 2, (uint32_t)kList)];
          blend(now, !done & now.in, c);
        }
      } else {
        for (uint32_t t = 0; t < steps; t++) {
          FwdPair p;
          p.evaluate(my_list[t], pixel_bit, s0, s1, px, py);
          const bool pass1 = !done & p.in;
          if (COUNT) {
            const uint64_t b1 = __ballot(pass1);
            pcount[0]++;
            if (!b1) continue;
            pcount[1]++;
            pcount[2] += (uint32_t)__popcll(b1);
          } else if (__builtin_amdgcn_ballot_w64(pass1) == 0) {
            continue;
          }
          const float4 c = at_bytes(s2, p.k16);
          p.exponent(tab);
          blend(p, pass1, c);
        }
      }
      if (last != 0xffffffffu) nc = b0 - start + (last >> 4) + 1;
    }
  }
  if (valid) {
    const size_t pix = tg.pix0 + (size_t)(ti.gy0 + j) * tg.width + ti.gx0 + i;
    image[pix * 3 + 0] = c0 + T * bg0;
    image[pix * 3 + 1] = c1 + T * bg1;
    image[pix * 3 + 2] = c2 + T * bg2;
    final_t[pix] = T;
    n_contrib[pix] = nc;
  }
  if (COUNT) flush_counts(pairs, kFwdVisits, pcount, 5);
  if (!PERSIST) break;
  }
}

// Per-pixel backward state (PixelBack, src/rasterize.rs:345-350).
struct PixBack {
  float t, acc0, acc1, acc2, last_alpha, lc0, lc1, lc2;
  float d0, d1, d2, bg_dot, t_final;
  uint32_t last;
};

// Terms of one (entry, pixel) pair, src/rasterize.rs:404-445, in predicated form: `act`
// says the pixel is inside the entry's rectangle and before its last contributor.
// Returns whether any lane of the wave contributes; v[] holds the slot terms (zero for
// lanes that do not), and the pixel state advances only on contributing lanes.  The
// reference's expressions and correctly rounded divisions: the ordered backward is bitwise.
// bg (uniform over the wave): the background term is not a zero for every lane.
__device__ __forceinline__ bool pair_terms(PixBack& s, bool act, float4 r0, float4 r1, float4 r2,
                                           float px, float py, const uint64_t* tab, bool bg,
                                           float v[kSlots]) {
#pragma unroll
  for (int q = 0; q < kSlots; q++) v[q] = 0.0f;
  const float dx = px - r0.x;
  const float dy = py - r0.y;
  const float sigma = (r0.z * dx * dx + r1.x * dy * dy) + r0.w * dx * dy;  // halved A, C
  const bool p1 = act & !((sigma < 0.0f) | (sigma > r1.z));
  if (__builtin_amdgcn_ballot_w64(p1) == 0) return false;
  const float G = expf_walk_tab(-sigma, tab);  // used where 0 <= sigma <= sigma_max
  const float o = r1.y;
  const float og = o * G;
  const bool p2 = p1 & !(og < kAlphaMin);
  const float alpha = rmin(og, kAlphaMax);
  const float t = s.t / (1.0f - alpha);
  const float a0 = s.last_alpha * s.lc0 + (1.0f - s.last_alpha) * s.acc0;
  const float a1 = s.last_alpha * s.lc1 + (1.0f - s.last_alpha) * s.acc1;
  const float a2 = s.last_alpha * s.lc2 + (1.0f - s.last_alpha) * s.acc2;
  float dalpha = 0.0f;
  dalpha += (r2.y - a0) * s.d0;
  dalpha += (r2.z - a1) * s.d1;
  dalpha += (r2.w - a2) * s.d2;
  dalpha *= t;
  // without a background the term is a zero, whose addition no sum sees
  if (bg) dalpha += (-s.t_final / (1.0f - alpha)) * s.bg_dot;
  const bool p3 = p2 & (og < kAlphaMax);
  const float dgauss = o * dalpha;
  const float dsigma = -dgauss * G;
  const float ddx = dsigma * ((2.0f * r0.z) * dx + r0.w * dy);
  const float ddy = dsigma * (r0.w * dx + (2.0f * r1.x) * dy);
  v[6] = p2 ? alpha * t * s.d0 : 0.0f;
  v[7] = p2 ? alpha * t * s.d1 : 0.0f;
  v[8] = p2 ? alpha * t * s.d2 : 0.0f;
  v[5] = p3 ? G * dalpha : 0.0f;
  v[0] = p3 ? -ddx : 0.0f;
  v[1] = p3 ? -ddy : 0.0f;
  v[2] = p3 ? dsigma * 0.5f * dx * dx : 0.0f;
  v[3] = p3 ? dsigma * dx * dy : 0.0f;
  v[4] = p3 ? dsigma * 0.5f * dy * dy : 0.0f;
  v[9] = p3 ? fabsf(ddx) : 0.0f;
  v[10] = p3 ? fabsf(ddy) : 0.0f;
  if (p2) {
    s.t = t;
    s.acc0 = a0;
    s.acc1 = a1;
    s.acc2 = a2;
    s.lc0 = r2.y;
    s.lc1 = r2.z;
    s.lc2 = r2.w;
    s.last_alpha = alpha;
  }
  return true;
}

// v as seen through a DPP control within each 16-lane row (every lane has a source).  The
// compiler folds the move into the instruction that consumes it.
template <int CTRL>
__device__ __forceinline__ float dpp_row(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Sum over each 16-lane row by a rotate butterfly: every lane ends with its row's sum.
__device__ __forceinline__ float row_allsum16(float v) {
  v += dpp_row<0x121>(v);  // row_ror:1
  v += dpp_row<0x122>(v);  // row_ror:2
  v += dpp_row<0x124>(v);  // row_ror:4
  v += dpp_row<0x128>(v);  // row_ror:8
  return v;
}

// Sums of nine values over each 16-lane row: lanes 2m and 2m+1 of the row end with the sum
// of v[m] for m < 8, except that lane 15 ends with the sum of v[8].  v[0..7] go through a
// reduce-scatter whose steps pair a lane with lane ^ {8, 7, 2, 1}; the two partners keep
// complementary halves of their values (chosen by bit 3, 2, 1 of the lane) and add the half
// the other sends.  The four masks span all 16 lanes, so every sum covers the row; the order
// of the additions is fixed.  v[8] goes through row_allsum16's butterfly.
//
// The first two steps select by lane bits 3 and 2, which are exactly the DPP banks (lanes
// 4k .. 4k + 3 of a row): two bank-masked DPP adds, each writing half of the row, give
// x + x(partner) on one half and y + y(partner) on the other.  The compiler does not form
// masked DPP adds, so the whole reduction is written out.  A DPP read needs two wait states
// after the VALU write of its source: v[8]'s steps stand between the others' for that, and
// two s_nops cover the inputs and the last step (six blocks with a pair of s_nops each spent
// 12 more issue slots per step of the walk).
// upper: mask of the lanes with bit 1 set; last: of the rows' lanes 15.
__device__ __forceinline__ float row_sums9(float v0, float v1, float v2, float v3, float v4,
                                           float v5, float v6, float v7, float v8,
                                           uint64_t upper, uint64_t last) {
  asm volatile(
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"  // banks 0-1: v0
      "v_add_f32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"  // banks 2-3: v4
      "v_add_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %1, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %2, %2, %2 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %2, %6, %6 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %3, %3, %3 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %3, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %8, %8, %8 row_ror:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %0, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %8, %8, %8 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_add_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %1, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %8, %8, %8 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %4, %1, %0, %9\n\t"   // the half to send
      "v_cndmask_b32_e64 %5, %0, %1, %9\n\t"   // the half to keep
      "v_add_f32_dpp %8, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_add_f32_dpp %0, %4, %5 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %0, %0, %8, %10"
      : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3), "+v"(v4), "+v"(v5), "+v"(v6), "+v"(v7), "+v"(v8)
      : "s"(upper), "s"(last));
  return v0;
}

// pair_terms in the tree-reduced form, rearranged for fewer instructions.  Equal up to
// rounding; the decisions (sigma range, alpha_min, alpha_max) are the exact ones, so the
// walk visits the same pairs as the forward:
//  * one hardware reciprocal y (1 ulp) of d = 1 - alpha serves both divisions by d.  The
//    transmittance, which the walk divides again at every contributor, takes one residual
//    correction, t = q + (s.t - q d) y with q = s.t y and the residual exact in an fma: the
//    error before the final rounding is O(ulp^2), so t is the correctly rounded quotient
//    (the reference's) but for inputs within 2^-45 of a rounding midpoint, and no bias
//    of the reciprocal builds up along the walk.  The background term's T_final / d takes
//    the same correction; with a black background (BG = false) that term is zero and is
//    left out;
//  * the accumulated colour behind the next contributor is updated eagerly,
//    A <- A + alpha (c - A), the reference's last_alpha * last_color + (1 - last_alpha) * acc
//    (src/rasterize.rs:420-428) evaluated one entry earlier;
//  * with q = dL/dsigma the slots 0-4 become the per-pixel products q dx, q dy, q dx^2,
//    q dx dy, q dy^2; the entry's conic turns the sums into dL/dmean and 0.5 scales the
//    diagonal conic slots once per entry, when the batch's slots are written;
//  * products with a zero factor stand in for the per-slot selects.
// The pixel state uses acc0..2 for A; lc and last_alpha are unused.  Returns the row sums of
// the slot terms as row_sums9 leaves them in the lanes (with ABS, slots 9 and 10 in the rows'
// lanes 13 and 11).
// The step in two parts: evaluate() and exponent() depend on the pair alone, sums() on the
// pixel's state.
template <bool ABS>
struct BwdPair {
  bool in;  // the pixel is a candidate of the entry and 0 <= sigma <= sigma_max
  float dx, dy, sigma, o, G;
  __device__ __forceinline__ void evaluate(bool act, float4 r0, float4 r1, float px, float py) {
    dx = px - r0.x;
    dy = py - r0.y;
    sigma = (r0.z * dx * dx + r1.x * dy * dy) + r0.w * dx * dy;  // halved A, C
    in = act & !((sigma < 0.0f) | (sigma > r1.z));
    o = r1.y;
  }
  __device__ __forceinline__ void exponent(const uint64_t* tab) {
    G = expf_walk_tab(-sigma, tab);  // used where 0 <= sigma <= sigma_max
  }
  // r0z, r0w, r1x: the (halved) conic, read with ABS only.  passing (COUNT): += passing pairs.
  template <bool COUNT>
  __device__ __forceinline__ float sums(PixBack& s, float4 r2, bool bg, float r0z, float r0w,
                                        float r1x, uint32_t* passing) const {
    const float og = o * G;
    const bool p2 = in & !(og < kAlphaMin);
    const bool p3 = p2 & (og < kAlphaMax);
    if (COUNT) *passing += (uint32_t)__popcll(__ballot(p2));
    const float alpha = rmin(og, kAlphaMax);
    const float den = 1.0f - alpha;
    const float inv = __builtin_amdgcn_rcpf(den);
    const float q0 = s.t * inv;
    const float t = fmaf(fmaf(-q0, den, s.t), inv, q0);
    const float e0 = r2.y - s.acc0, e1 = r2.z - s.acc1, e2 = r2.w - s.acc2;
    float dalpha = e0 * s.d0;
    dalpha = fmaf(e1, s.d1, dalpha);
    dalpha = fmaf(e2, s.d2, dalpha);
    if (bg) {  // uniform: a kernel argument
      const float f0 = s.t_final * inv;
      const float tf = fmaf(fmaf(-f0, den, s.t_final), inv, f0);
      dalpha = fmaf(dalpha, t, -tf * s.bg_dot);
    } else {
      dalpha *= t;
    }
    const float q = p3 ? -(o * dalpha) * G : 0.0f;
    const float w = p2 ? alpha * t : 0.0f;
    s.t = p2 ? t : s.t;
    s.acc0 = p2 ? fmaf(alpha, e0, s.acc0) : s.acc0;
    s.acc1 = p2 ? fmaf(alpha, e1, s.acc1) : s.acc1;
    s.acc2 = p2 ? fmaf(alpha, e2, s.acc2) : s.acc2;
    const float qdx = q * dx, qdy = q * dy;
    constexpr uint64_t kUpper = 0xccccccccccccccccull, kLast = 0x8000800080008000ull;
    float out = row_sums9(qdx, qdy, qdx * dx, qdx * dy, qdy * dy, p3 ? G * dalpha : 0.0f,
                          w * s.d0, w * s.d1, w * s.d2, kUpper, kLast);
    if (ABS) {
      const float e9 = row_allsum16(fabsf(fmaf(2.0f * r0z, qdx, r0w * qdy)));
      const float e10 = row_allsum16(fabsf(fmaf(r0w, qdx, (2.0f * r1x) * qdy)));
      const uint32_t l16 = threadIdx.x & 15u;
      out = l16 == 13 ? e9 : out;
      out = l16 == 11 ? e10 : out;
    }
    return out;
  }
};

// A pixel's state at the start of the backward walk.  valid: inside the image.
__device__ __forceinline__ PixBack pixel_back(const TileGeom& tg, uint32_t i, uint32_t j,
                                              bool valid, float bg0, float bg1, float bg2,
                                              const float* __restrict__ final_t,
                                              const uint32_t* __restrict__ n_contrib,
                                              const float* __restrict__ dimage) {
  PixBack s;
  s.acc0 = s.acc1 = s.acc2 = 0.0f;
  s.lc0 = s.lc1 = s.lc2 = 0.0f;
  s.last_alpha = 0.0f;
  s.t = 1.0f;
  s.t_final = 1.0f;
  s.d0 = s.d1 = s.d2 = 0.0f;
  s.bg_dot = 0.0f;
  s.last = 0;
  if (valid) {
    const size_t pix = tg.pix0 + (size_t)(tg.ti.gy0 + j) * tg.width + tg.ti.gx0 + i;
    s.d0 = dimage[pix * 3 + 0];
    s.d1 = dimage[pix * 3 + 1];
    s.d2 = dimage[pix * 3 + 2];
    s.bg_dot = bg0 * s.d0 + bg1 * s.d1 + bg2 * s.d2;
    s.last = n_contrib[pix];
    s.t_final = final_t[pix];
    s.t = s.t_final;
  }
  return s;
}

// The tree-reduced backward: 16-lane row sums by DPP (row_sums9), an entry's row partials
// summed in a fixed order.  Bound by VALU issue (about 100 instructions per walk step).  Of
// the LDS partials only those that svisit names are written and read: clearing all 16 rows of
// every entry and summing them took as many instructions as a fifth of the walk.  With that,
// the list words (as in the forward) and the row sums in one block: 10k Gaussians, 256x256,
// 139 -> 123 us; with records prefetched too, 1M Gaussians, 1920x1080: 471 -> 428 us.
// ABS: also accumulate the AbsGS slots (9, 10).  B: entries per LDS batch.  ROWS: every
// 16-lane row walks its own entry list; otherwise the wave walks the entries that reach any
// of its rows (the same sums either way).  COUNT: also count pairs into `pairs`
// (PairCounter).
// FEW: for launches with few tiles (kFewTilesBwd); rows only.
template <bool ABS, int B, bool BATCH, bool PERSIST, bool ROWS, bool COUNT = false,
          bool FEW = false>
__global__ void __launch_bounds__(256) raster_bwd_kernel(
    const float4* __restrict__ rec, const uint32_t* __restrict__ tile_start,
    const uint32_t* __restrict__ order,
    const uint32_t* __restrict__ sorted_gauss, const uint32_t* __restrict__ sorted_entry,
    uint32_t num_tiles, uint32_t tiles_x, uint32_t W, uint32_t H, float bg0, float bg1,
    float bg2, const float* __restrict__ final_t, const uint32_t* __restrict__ n_contrib,
    const float* __restrict__ dimage, float* __restrict__ slots, BatchDev bd,
    uint32_t* __restrict__ counter, unsigned long long* __restrict__ pairs) {
  static_assert(B <= 32 || (B == 64 && ROWS), "a list is built by half a wave, or by a wave");
  // words per entry in `slots` and per row partial: the absolute sums (9, 10) only when asked
  constexpr uint32_t SS = ABS ? kSlots : 9;
  __shared__ uint64_t tab[32];
  __shared__ float4 s0[B], s1[B], s2[B];
  __shared__ uint32_t srect[B], sentry[B];
  __shared__ __align__(4) uint8_t svisit[B][4];  // per entry and wave: the rows that wrote a partial
  __shared__ uint32_t slist[16][B + 1];  // per (wave, row): its entries, back to front
  __shared__ uint32_t smax_last;
  __shared__ uint32_t s_tile;
  // Partials of the batch, [entry][wave, row][word]; only those named by svisit are written
  // and read (an entry reaches 2 to 3 of a tile's 16 rows on average).
  __shared__ float red[B * 16 * SS];
  // whether the background term (T_final bg . dL) can be non-zero for a finite dL
  const bool bg_any = (bg0 != 0.0f) | (bg1 != 0.0f) | (bg2 != 0.0f);
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Table[threadIdx.x];
  if (FEW && threadIdx.x < 16) slist[threadIdx.x][B] = 0u;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4;
  const uint32_t l16 = lane & 15u;
  const uint32_t pixel_bit = 0x10000u << l16;
  // the slot whose row sum this lane holds after a step, if it writes one: even lane 2m slot
  // m, lane 15 slot 8, lanes 13 and 11 the AbsGS slots 9 and 10
  const bool even = (l16 & 1u) == 0;
  const bool writer = even | (l16 == 15) | (ABS & ((l16 == 13) | (l16 == 11)));
  const uint32_t wslot = even ? (l16 >> 1) : (l16 == 15 ? 8u : (l16 == 13 ? 9u : 10u));
  for (;;) {
  const uint32_t tile = next_tile<PERSIST>(counter, &s_tile, order, num_tiles);
  if (tile >= num_tiles) break;
  if (threadIdx.x == 0) smax_last = 0;
  const TileGeom tg = tile_geom<BATCH>(tile, tiles_x, W, H, bd);
  const TileInfo ti = tg.ti;
  uint32_t i, j;
  tile_pixel(threadIdx.x, &i, &j);
  const bool valid = i < ti.w && j < ti.h;
  const float px = (float)(ti.gx0 + i) + 0.5f;
  const float py = (float)(ti.gy0 + j) + 0.5f;
  PixBack s = pixel_back(tg, i, j, valid, bg0, bg1, bg2, final_t, n_contrib, dimage);
  const uint32_t start = tile_start[tile], end = tile_start[tile + 1];
  const uint32_t count = end - start;
  uint32_t pcount[4] = {0, 0, 0, 0};
  __syncthreads();
  if (valid && s.last > 0) atomicMax(&smax_last, s.last);
  __syncthreads();
  const uint32_t kmax = min(smax_last, count);
  // Entries no pixel reaches get zero slots.
  for (uint32_t q = kmax * SS + threadIdx.x; q < count * SS; q += blockDim.x) {
    const uint32_t k = q / SS;
    slots[(size_t)sorted_entry[start + k] * SS + q % SS] = 0.0f;
  }
  // the last contributor of any pixel of each 16-lane row of this wave
  uint32_t row_last[4];
  {
    uint32_t m = valid ? s.last : 0u;
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d, 64));
#pragma unroll
    for (int r = 0; r < 4; r++) row_last[r] = (uint32_t)__builtin_amdgcn_readlane((int)m, 16 * r);
  }
  const uint32_t wave_last = max(max(row_last[0], row_last[1]), max(row_last[2], row_last[3]));
  // Batches walk [0, kmax) from the back.  A batch's records are loaded while the batch behind
  // it is summed, their Gaussians and entry ids while it is walked (lanes past a batch's end
  // repeat its last entry).
  StagedRecord sr{};
  uint32_t next_g = 0, entry_id = 0, next_id = 0;
  const auto batch_index = [&](int32_t h) {  // of the batch that ends at h
    const int32_t l = max(h - B, 0);
    return start + (uint32_t)min(l + (int32_t)threadIdx.x, h - 1);
  };
  if (threadIdx.x < B && kmax > 0) {
    const uint32_t at = batch_index((int32_t)kmax);
    next_g = sorted_gauss[at];
    entry_id = sorted_entry[at];
    sr = load_record(rec, next_g);
  }
  for (int32_t hi = (int32_t)kmax; hi > 0; hi -= B) {
    const int32_t lo = max(hi - B, 0);
    const uint32_t cnt = (uint32_t)(hi - lo);
    __syncthreads();
    if (threadIdx.x < B) {
      s0[threadIdx.x] = half_conic0(sr.a);
      s1[threadIdx.x] = half_conic1(sr.b);
      s2[threadIdx.x] = sr.c;
      srect[threadIdx.x] = entry_rect(sr.a, sr.b, sr.c, ti);
      sentry[threadIdx.x] = entry_id;
      if (lo > 0) {
        const uint32_t at = batch_index(lo);
        next_g = sorted_gauss[at];
        next_id = sorted_entry[at];
      }
    }
    __syncthreads();
    // Each 16-lane row walks, back to front, only the batch entries that reach its 4x4
    // sub-block and precede the row's last contributor; the four rows of a wave walk
    // their own lists side by side.  One entry per lane; with batches of up to 32, lanes 0-31
    // build the lists of rows 0 and 1, lanes 32-63 those of rows 2 and 3.
    constexpr uint32_t kHalf = B <= 32 ? 32 : 64;
    const uint32_t kl = lane % kHalf, half = lane / kHalf;
    const uint32_t rc = kl < cnt ? srect[min(kl, (uint32_t)B - 1u)] : 0u;
    uint32_t steps = 0, visit = 0;
    uint64_t wave_todo = 0;  // !ROWS: the wave's entries, walked from the top bit down
    if (ROWS) {
#pragma unroll
      for (uint32_t r = 0; r < kHalf / 16; r++) {
        const uint32_t q = half * 2 + r;  // the row
        const uint32_t last = half ? row_last[(r + 2) % 4] : row_last[r];
        const uint32_t pm = lo + kl < last ? row_mask(rc, wave, q) : 0u;
        const uint64_t m2 = __ballot(pm != 0);
        uint64_t m = m2;
        if (kHalf == 32) m = half ? m2 >> 32 : m2 & 0xffffffffull;
        const uint32_t len = (uint32_t)__popcll(m);
        uint32_t* list = slist[wave * 4 + q];
        // entry kl sits behind the later entries of the batch
        if (pm) list[__popcll(m >> kl) - 1] = (pm << 16) | (kl << 4);
        if (kl >= len && kl < (uint32_t)B) list[kl] = 0u;  // past the end: no entry
        if (pm) visit |= 1u << r;
        steps = max(steps, kHalf == 32 ? max((uint32_t)__popc((uint32_t)m2),
                                             (uint32_t)__popc((uint32_t)(m2 >> 32)))
                                       : len);
      }
      if (kHalf == 32) visit |= (uint32_t)__shfl((int)visit, (int)(kl + 32), 64) << 2;
    } else {
      const bool on = lane < cnt && lo + lane < wave_last && wave_touches(rc, wave);
      wave_todo = __ballot(on);
      steps = (uint32_t)__popcll(wave_todo);
      visit = on ? 0xfu : 0u;
    }
    if (lane < cnt) svisit[lane][wave] = (uint8_t)visit;
    // the lists are written and read by this wave only
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const uint32_t* my_list = slist[wave * 4 + row];
    const uint32_t last16 = s.last > (uint32_t)lo ? min(s.last - lo, (uint32_t)B) << 4 : 0u;
    const uint32_t my_red = (wave * 4 + row) * SS + wslot;
    if (FEW) {
      // the pair of the next step is evaluated beside the sums of this one
      uint32_t le = my_list[0], next = my_list[1];
      BwdPair<ABS> p;
      const auto prepare = [&] {
        const uint32_t k16 = le & 0xffffu;
        p.evaluate(((le & pixel_bit) != 0) & (k16 < last16), at_bytes(s0, k16), at_bytes(s1, k16),
                   px, py);
        p.exponent(tab);
      };
      prepare();
      for (uint32_t t = 0; t < steps; t++) {
        const BwdPair<ABS> now = p;
        const uint32_t k16 = le & 0xffffu;
        const bool has = le != 0;
        const float4 r2 = at_bytes(s2, k16);
        float r0z = 0, r0w = 0, r1x = 0;
        if (ABS) {
          const float4 r0 = at_bytes(s0, k16);
          r0z = r0.z;
          r0w = r0.w;
          r1x = at_bytes(s1, k16).x;
        }
        le = next;
        next = my_list[min(t + 2, (uint32_t)B)];
        prepare();
        // the sums count if some lane evaluates the pair, as below: a factor of zero leaves a
        // gradient that is not finite in them
        const bool any = __builtin_amdgcn_ballot_w64(now.in) != 0;
        const float sums = now.template sums<false>(s, r2, bg_any, r0z, r0w, r1x, nullptr);
        const float out = any ? sums : 0.0f;
        if (has & writer) red[k16 * SS + my_red] = out;
      }
    } else {
      for (uint32_t t = 0; t < steps; t++) {
        uint32_t k16;
        bool has = true, act;
        if (ROWS) {
          const uint32_t le = my_list[t];
          k16 = le & 0xffffu;
          has = le != 0;
          act = ((le & pixel_bit) != 0) & (k16 < last16);
        } else {
          const uint32_t kk = 63u - (uint32_t)__builtin_clzll(wave_todo);
          wave_todo &= ~(1ull << kk);
          k16 = kk << 4;
          act = (k16 < last16) & in_rect(srect[kk], i, j);
        }
        BwdPair<ABS> p;
        const float4 r0 = at_bytes(s0, k16), r1 = at_bytes(s1, k16);
        p.evaluate(act, r0, r1, px, py);
        float out = 0.0f;
        const uint64_t b1 = __builtin_amdgcn_ballot_w64(p.in);
        if (COUNT) pcount[0]++;
        if (b1) {
          if (COUNT) {
            pcount[1]++;
            pcount[2] += (uint32_t)__popcll(b1);
          }
          const float4 r2 = at_bytes(s2, k16);
          p.exponent(tab);
          out = p.template sums<COUNT>(s, r2, bg_any, r0.z, r0.w, r1.x, &pcount[3]);
        }
        if (has & writer) red[k16 * SS + my_red] = out;
      }
    }
    __syncthreads();
    entry_id = next_id;
    // assigned on every path: the registers are free during the walk
    sr = StagedRecord{};
    if (threadIdx.x < B) sr = load_record(rec, next_g);
    // Sum the batch's partials and write its slots: 16 lanes per entry, lane = slot.
    const uint32_t slot = threadIdx.x & 15u;
    for (uint32_t e0 = 0; e0 < cnt; e0 += 16) {
      const uint32_t kk = e0 + (threadIdx.x >> 4);
      if (kk < cnt && slot < SS) {
        const float4 a = s0[kk], b = s1[kk];
        const uint32_t v = *reinterpret_cast<const uint32_t*>(svisit[kk]);
        uint32_t rows =
            (v & 0xfu) | ((v >> 4) & 0xf0u) | ((v >> 8) & 0xf00u) | ((v >> 12) & 0xf000u);
        const float* p = &red[kk * 16 * SS + slot];
        float acc = 0.0f;
        while (rows) {
          acc += p[(uint32_t)__builtin_ctz(rows) * SS];
          rows &= rows - 1;
        }
        // the products' sums: slots 0, 1 combine both position sums with the conic
        const float other = dpp_row<0xb1>(acc);  // lane ^ 1
        if (slot == 0)
          acc = -fmaf(2.0f * a.z, acc, a.w * other);
        else if (slot == 1)
          acc = -fmaf(a.w, other, (2.0f * b.x) * acc);
        else if (slot == 2 || slot == 4)
          acc *= 0.5f;
        slots[(size_t)sentry[kk] * SS + slot] = acc;
      }
    }
  }
  if (COUNT) flush_counts(pairs, kBwdVisits, pcount, 4);
  if (!PERSIST) break;
  }
}

// The ordered backward: an entry's per-pixel terms are staged in LDS and summed one by one
// in row-major order.  Only the pixels of the entry's rectangle have terms (the others are
// exact zeros, which a sum that starts at +0 does not see), so the staging is packed: the
// entries of a group, as many as fit kTerms pixels, lie one after the other, and a lane
// sums one slot of one entry over the entry's own pixels.  Only the waves whose 8x8 block the
// rectangle reaches evaluate it.
//
// FEW (launches with few tiles, kFewTilesOrd): bound by the latency of the walk and of the
// sums' chains of up to 256 additions, so they overlap: a fifth wave sums a group while the
// four of the pixels walk the next one into the other half of the staging, and loads the next
// batch's records; a group holds four full tiles.  Otherwise the chip is filled by other
// workgroups, walk and sums take turns and the staging is kept small (two full tiles).  In us,
// FEW / otherwise / all 256 pixels of 8 entries staged at a time, as it was: 130 tiles of a
// grown model (most entries cover their tiles) 511 / 680 / 1279, 256 tiles 177 / 229 / 403,
// 4293 tiles 2060 / 875 / 4526, 8160 tiles 2401 / 750 / 5785.  FEW / otherwise on the scenes of
// kFewTilesFwd: 675 tiles 187 / 244 and 593 / 814, 900 tiles 204 / 262 and 507 / 700, 1120 tiles
// 245 / 246 and 543 / 756, 1271 tiles 262 / 206 and 497 / 696, 1600 tiles 336 / 269 and 630 / 872:
// the line lies where neither is slower.  (The slots' rows lie four words apart modulo the LDS
// banks and are read 16 bytes at a time, the next ones beside the additions; in step and one word
// at a time it was 940 at 130 tiles and 1217 at 8160.)
template <bool ABS, bool BATCH, bool PERSIST, bool FEW>
__global__ void __launch_bounds__(FEW ? 320 : 256) raster_bwd_ordered_kernel(
    const float4* __restrict__ rec, const uint32_t* __restrict__ tile_start,
    const uint32_t* __restrict__ order,
    const uint32_t* __restrict__ sorted_gauss, const uint32_t* __restrict__ sorted_entry,
    uint32_t num_tiles, uint32_t tiles_x, uint32_t W, uint32_t H, float bg0, float bg1,
    float bg2, const float* __restrict__ final_t, const uint32_t* __restrict__ n_contrib,
    const float* __restrict__ dimage, float* __restrict__ slots, BatchDev bd,
    uint32_t* __restrict__ counter) {
  constexpr uint32_t SS = ABS ? kSlots : 9;
  constexpr int B = kOrdBatch;
  constexpr uint32_t kTerms = FEW ? 1024 : 512;  // pixel terms per slot staged at a time
  constexpr uint32_t kRow = kTerms + 4;          // words per slot: slots apart in the LDS banks
  static_assert(B < 64 && kTerms >= 256, "one wave scans a batch; a group holds an entry");
  // FEW: two batches and two groups, one being walked, the other summed or loaded
  constexpr int kHalves = FEW ? 2 : 1;
  __shared__ uint64_t tab[32];
  __shared__ float4 s0[kHalves][B], s1[kHalves][B], s2[kHalves][B];
  __shared__ uint32_t srect[kHalves][B], sentry[kHalves][B];
  __shared__ uint32_t spre[kHalves][B + 1];  // staging words of the batch entries before each one
  __shared__ uint32_t smax_last;
  __shared__ uint32_t s_tile;
  __shared__ __align__(16) float terms[kHalves][SS * kRow + 16];  // (a sum reads 16 words ahead)
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Table[threadIdx.x];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool walker = !FEW || wave < 4;  // uniform over the wave
  for (;;) {
  const uint32_t tile = next_tile<PERSIST>(counter, &s_tile, order, num_tiles);
  if (tile >= num_tiles) break;
  if (threadIdx.x == 0) smax_last = 0;
  const TileGeom tg = tile_geom<BATCH>(tile, tiles_x, W, H, bd);
  const TileInfo ti = tg.ti;
  uint32_t i, j;
  tile_pixel(threadIdx.x & 255u, &i, &j);
  const bool valid = walker && i < ti.w && j < ti.h;
  const float px = (float)(ti.gx0 + i) + 0.5f;
  const float py = (float)(ti.gy0 + j) + 0.5f;
  PixBack s = pixel_back(tg, i, j, valid, bg0, bg1, bg2, final_t, n_contrib, dimage);
  // whether the background term of some pixel of the wave is not a zero
  const bool bg = __any(!(s.bg_dot == 0.0f) || !(fabsf(s.t_final) < INFINITY));
  const uint32_t start = tile_start[tile], end = tile_start[tile + 1];
  const uint32_t count = end - start;
  __syncthreads();
  if (valid && s.last > 0) atomicMax(&smax_last, s.last);
  __syncthreads();
  const uint32_t kmax = min(smax_last, count);
  // Entries no pixel reaches get zero slots.
  for (uint32_t q = kmax * SS + threadIdx.x; q < count * SS; q += blockDim.x) {
    const uint32_t k = q / SS;
    slots[(size_t)sorted_entry[start + k] * SS + q % SS] = 0.0f;
  }
  // (one wave) the batch of entries [lo, lo + cnt) into half `h`
  const auto stage = [&](uint32_t h, uint32_t lo, uint32_t cnt) {
    uint32_t area = 0;
    if (lane < cnt) {
      const uint32_t at = start + lo + lane;
      const StagedRecord r = load_record(rec, sorted_gauss[at]);
      sentry[h][lane] = sorted_entry[at];
      s0[h][lane] = half_conic0(r.a);
      s1[h][lane] = half_conic1(r.b);
      s2[h][lane] = r.c;
      const uint32_t rc = entry_rect(r.a, r.b, r.c, ti);
      srect[h][lane] = rc;
      // whole groups of four, for 16-byte reads
      area = ((uint32_t)__popc(rc & 0xffffu) * (uint32_t)__popc(rc >> 16) + 3u) & ~3u;
    }
    uint32_t pre = area;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = (uint32_t)__shfl_up((int)pre, d, 64);
      if (lane >= (uint32_t)d) pre += o;
    }
    if (lane <= cnt) spre[h][lane] = pre - area;
  };
  // (lanes q0, q0 + step, ...) the slots of group [g0, g1) of the batch in half `h`, staged in
  // terms[tb]
  const auto sum_group = [&](uint32_t h, uint32_t g0, uint32_t g1, uint32_t tb, uint32_t q0,
                             uint32_t step) {
    const uint32_t p0 = spre[h][g0];
    for (uint32_t q = q0; q < (g1 - g0) * SS; q += step) {
      const uint32_t kk = g0 + q / SS, slot = q % SS;
      const uint32_t rc = srect[h][kk];
      const uint32_t n = (uint32_t)__popc(rc & 0xffffu) * (uint32_t)__popc(rc >> 16);
      const float4* p =
          reinterpret_cast<const float4*>(&terms[tb][slot * kRow + (spre[h][kk] - p0)]);
      // the additions stay in order; the next eight terms are read beside them
      float acc = 0.0f;
      float4 x = p[0], y = p[1];  // (within the array whatever n is)
      uint32_t t = 0;
      for (; t + 8 <= n; t += 8) {
        const float4 x0 = x, y0 = y;
        x = p[t / 4 + 2];
        y = p[t / 4 + 3];
        acc += x0.x;
        acc += x0.y;
        acc += x0.z;
        acc += x0.w;
        acc += y0.x;
        acc += y0.y;
        acc += y0.z;
        acc += y0.w;
      }
      const float rest[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
      for (uint32_t u = 0; u < 7; u++)
        if (t + u < n) acc += rest[u];
      slots[(size_t)sentry[h][kk] * SS + slot] = acc;
    }
  };
  uint32_t h = 0, tb = 0;                        // batch half, staging half
  uint32_t last_h = 0, last_g0 = 0, last_g1 = 0;  // the group walked before this one (none: g1 = 0)
  if (FEW) {
    if (!walker && kmax > 0) stage(0, max((int32_t)kmax - B, 0), min(kmax, (uint32_t)B));
    __syncthreads();
  }
  for (int32_t hi = (int32_t)kmax; hi > 0; hi -= B) {
    const int32_t lo = max(hi - B, 0);
    const uint32_t cnt = (uint32_t)(hi - lo);
    if (!FEW) {
      __syncthreads();
      if (wave == 0) stage(0, (uint32_t)lo, cnt);
      __syncthreads();
    }
    // groups of entries from the back, each the longest that fits the staging
    const uint32_t my_pre = spre[h][min(lane, cnt)];
    for (uint32_t g1 = cnt; g1 > 0;) {
      const uint32_t p1 = spre[h][g1];
      const uint64_t fits = __ballot(lane < g1 && p1 - my_pre <= kTerms);
      const uint32_t g0 = (uint32_t)__builtin_ctzll(fits);  // entry g1 - 1 fits (<= 256 pixels)
      if (walker) {
        const uint32_t p0 = spre[h][g0];
        uint64_t todo = __ballot(lane >= g0 && lane < g1 &&
                                 wave_touches(srect[h][min(lane, cnt - 1)], wave));
        while (todo) {
          const uint32_t kk = 63u - (uint32_t)__builtin_clzll(todo);
          todo &= ~(1ull << kk);
          const uint32_t rc = srect[h][kk];
          const bool in = in_rect(rc, i, j);  // columns and rows are within the image
          float v[kSlots];
          pair_terms(s, valid & (lo + kk < s.last) & in, s0[h][kk], s1[h][kk], s2[h][kk], px, py,
                     tab, bg, v);
          if (in) {
            const uint32_t x0 = (uint32_t)__builtin_ctz(rc), y0 = (uint32_t)__builtin_ctz(rc >> 16);
            const uint32_t pos =
                spre[h][kk] - p0 + (j - y0) * (uint32_t)__popc(rc & 0xffffu) + (i - x0);
#pragma unroll
            for (int q = 0; q < (int)SS; q++) terms[tb][q * kRow + pos] = v[q];
          }
        }
      } else {
        if (last_g1) sum_group(last_h, last_g0, last_g1, tb ^ 1u, lane, 64);
        // the other half's batch is summed: the next batch goes there, once per batch
        if (g1 == cnt && lo > 0) stage(h ^ 1u, (uint32_t)max(lo - B, 0), min((uint32_t)lo, (uint32_t)B));
      }
      __syncthreads();
      if (FEW) {
        last_h = h;
        last_g0 = g0;
        last_g1 = g1;
        tb ^= 1u;
      } else {
        sum_group(0, g0, g1, 0, threadIdx.x, 256);
        __syncthreads();
      }
      g1 = g0;
    }
    if (FEW) h ^= 1u;
  }
  if (FEW && !walker && last_g1) sum_group(last_h, last_g0, last_g1, tb ^ 1u, lane, 64);
  if (!PERSIST) break;
  }
}

// Sum each row's slots over its entries in entry order (src/rasterize.rs:480-503).  One
// wave per 64 / NS consecutive rows, one lane per (row, slot): the rows' entries form one
// span, staged through LDS in windows with coalesced loads, and each lane adds its slot of
// its row's entries in order, so every sum keeps the reference's sequential order.  NS is
// the record width the backward wrote: 9, or 11 with the absolute sums (slots 9 and 10,
// into abs_grads).  A window of 128 entries holds the span of a wave's rows in the dense
// batched workload (about 100 entries) and keeps the workgroup's LDS at 4.6 KB (9 slots),
// so that LDS does not limit how many waves a CU holds (256 entries: 9.2 KB, about half).
constexpr uint32_t kReduceWindow = 128;  // entries staged per window

template <int NS>
__global__ void __launch_bounds__(64) reduce_slots_kernel(const uint32_t* __restrict__ entry_offset,
                                                          const float* __restrict__ slots,
                                                          uint32_t n,
                                                          splat_proj_grad* __restrict__ grads,
                                                          float* __restrict__ abs_grads,
                                                          const StepStatus* __restrict__ status) {
  constexpr uint32_t kRows = 64 / NS;
  constexpr uint32_t kLoads = 16;  // loads per lane in flight before their LDS stores
  __shared__ float sh[kReduceWindow * NS];
  if (status && status->abort) return;  // uniform
  const uint32_t lane = threadIdx.x;
  const uint32_t r0 = blockIdx.x * kRows, rl = lane / NS, k = lane % NS;
  const uint32_t row = r0 + rl;
  const bool live = rl < kRows && row < n;
  const uint32_t span0 = entry_offset[r0], span1 = entry_offset[min(r0 + kRows, n)];
  const uint32_t e0 = live ? entry_offset[row] : 0u, e1 = live ? entry_offset[row + 1] : 0u;
  float sum = 0.0f;
  for (uint32_t c0 = span0; c0 < span1; c0 += kReduceWindow) {
    const uint32_t words = (min(c0 + kReduceWindow, span1) - c0) * NS;
    const float* src = slots + (size_t)c0 * NS;
    __syncthreads();
    for (uint32_t q0 = 0; q0 < words; q0 += 64 * kLoads) {
      float t[kLoads];
#pragma unroll
      for (uint32_t u = 0; u < kLoads; u++) {
        const uint32_t q = q0 + u * 64 + lane;
        t[u] = src[min(q, words - 1)];  // in the window: no branch between the loads
      }
#pragma unroll
      for (uint32_t u = 0; u < kLoads; u++) {
        const uint32_t q = q0 + u * 64 + lane;
        if (q < words) sh[q] = t[u];
      }
    }
    __syncthreads();
    const uint32_t hi = min(e1, c0 + kReduceWindow);
    for (uint32_t e = max(e0, c0); e < hi; e++) sum += sh[(e - c0) * NS + k];
  }
  if (!live) return;
  // splat_proj_grad holds slots 0-8 in slot order
  if (k < 9)
    reinterpret_cast<float*>(grads + row)[k] = sum;
  else
    abs_grads[2 * (size_t)row + (k - 9)] = sum;
}

}  // namespace

namespace {

// Whether a launch of one view of T tiles, one workgroup each, takes the FEW kernel: only the
// default shape does, every other runs as given.
bool few_fwd(const RasterVariant& rv, unsigned T) {
  return rv.fwd_batch == 0 && !rv.persistent && T <= kFewTilesFwd;
}
bool few_bwd(const RasterVariant& rv, unsigned T) {
  return rv.bwd_batch == 0 && !rv.persistent && rv.rows && T <= kFewTilesBwd;
}

// Workgroups of a persistent launch: `per_cu` per compute unit.
unsigned persistent_grid(splat_ctx* ctx, unsigned per_cu, unsigned tiles) {
  int cus = 0;
  SPLAT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  return std::max(1u, std::min<unsigned>(tiles, (unsigned)cus * std::max(per_cu, 1u)));
}

template <int B, bool BATCH, bool PERSIST, bool FEW = false>
void fwd_go(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb, unsigned T,
            uint32_t width, uint32_t height, const float bg[3], float* image, float* final_t,
            uint32_t* n_contrib, const BatchDev& bd, uint32_t* counter, unsigned per_cu) {
  if (PERSIST) fill_u32(ctx, counter, kXcds, 0u);
  const unsigned grid = PERSIST ? persistent_grid(ctx, per_cu, T) : T;
  launch(ctx, "raster_fwd", raster_fwd_kernel<B, BATCH, PERSIST, false, FEW>, dim3(grid),
         dim3(256), 0,
         (const float4*)pb.rec, (const uint32_t*)bb.tile_start, (const uint32_t*)bb.tile_order,
         (const uint32_t*)bb.sorted_gauss, T, bb.tiles_x, width, height, bg[0], bg[1], bg[2],
         image, final_t, n_contrib, bd, counter, (unsigned long long*)nullptr);
}

template <bool ABS, int BF, bool BATCH, bool PERSIST, bool ROWS, bool FEW = false>
void bwd_go(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb, unsigned T,
            uint32_t width, uint32_t height, const float bg[3], const float* final_t,
            const uint32_t* n_contrib, const float* dimage, float* slots, const BatchDev& bd,
            uint32_t* counter, unsigned per_cu) {
  if (PERSIST) fill_u32(ctx, counter, kXcds, 0u);
  const unsigned grid = PERSIST ? persistent_grid(ctx, per_cu, T) : T;
  launch(ctx, "raster_bwd", raster_bwd_kernel<ABS, BF, BATCH, PERSIST, ROWS, false, FEW>, dim3(grid),
         dim3(256), 0, (const float4*)pb.rec, (const uint32_t*)bb.tile_start,
         (const uint32_t*)bb.tile_order, (const uint32_t*)bb.sorted_gauss,
         (const uint32_t*)bb.sorted_entry, T, bb.tiles_x, width,
         height, bg[0], bg[1], bg[2], final_t, n_contrib, dimage, slots, bd, counter,
         (unsigned long long*)nullptr);
}

template <bool ABS, bool BATCH, bool PERSIST>
void bwd_ordered_go(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb, unsigned T,
                    uint32_t width, uint32_t height, const float bg[3], const float* final_t,
                    const uint32_t* n_contrib, const float* dimage, float* slots,
                    const BatchDev& bd, uint32_t* counter, unsigned per_cu) {
  if (PERSIST) fill_u32(ctx, counter, kXcds, 0u);
  const unsigned grid = PERSIST ? persistent_grid(ctx, per_cu, T) : T;
  const auto go = [&](auto kernel, unsigned threads) {
    launch(ctx, "raster_bwd_ordered", kernel, dim3(grid), dim3(threads), 0,
           (const float4*)pb.rec, (const uint32_t*)bb.tile_start, (const uint32_t*)bb.tile_order,
           (const uint32_t*)bb.sorted_gauss, (const uint32_t*)bb.sorted_entry, T, bb.tiles_x,
           width, height, bg[0], bg[1], bg[2], final_t, n_contrib, dimage, slots, bd, counter);
  };
  if constexpr (!BATCH && !PERSIST) {
    if (T <= kFewTilesOrd)
      return go(raster_bwd_ordered_kernel<ABS, false, false, true>, 320);
  }
  go(raster_bwd_ordered_kernel<ABS, BATCH, PERSIST, false>, 256);
}

template <bool BATCH, bool PERSIST>
void fwd_pick(splat_ctx* ctx, const RasterVariant& rv, const ProjBuffers& pb,
              const BinBuffers& bb, unsigned T, uint32_t width, uint32_t height,
              const float bg[3], float* image, float* final_t, uint32_t* n_contrib,
              const BatchDev& bd, uint32_t* counter) {
  if constexpr (!BATCH && !PERSIST) {
    if (few_fwd(rv, T))
      return fwd_go<256, false, false, true>(ctx, pb, bb, T, width, height, bg, image, final_t,
                                             n_contrib, bd, counter, rv.per_cu);
  }
  switch (rv.fwd_batch) {
    case 32:
      return fwd_go<32, BATCH, PERSIST>(ctx, pb, bb, T, width, height, bg, image, final_t,
                                        n_contrib, bd, counter, rv.per_cu);
    case 128:
      return fwd_go<128, BATCH, PERSIST>(ctx, pb, bb, T, width, height, bg, image, final_t,
                                         n_contrib, bd, counter, rv.per_cu);
    case 256:  // one entry per lane: a whole batch per barrier pair
      return fwd_go<256, BATCH, PERSIST>(ctx, pb, bb, T, width, height, bg, image, final_t,
                                         n_contrib, bd, counter, rv.per_cu);
    default:
      return fwd_go<64, BATCH, PERSIST>(ctx, pb, bb, T, width, height, bg, image, final_t,
                                        n_contrib, bd, counter, rv.per_cu);
  }
}

template <bool BATCH, bool PERSIST, bool ROWS>
void bwd_rows_pick(splat_ctx* ctx, const RasterVariant& rv, const ProjBuffers& pb,
                   const BinBuffers& bb, unsigned T, uint32_t width, uint32_t height,
                   const float bg[3], const float* final_t, const uint32_t* n_contrib,
                   const float* dimage, float* slots, bool need_abs, const BatchDev& bd,
                   uint32_t* counter) {
  const unsigned pc = rv.per_cu;
  if constexpr (!BATCH && !PERSIST && ROWS) {
    if (few_bwd(rv, T)) {
      if (need_abs)
        return bwd_go<true, 64, false, false, true, true>(ctx, pb, bb, T, width, height, bg,
                                                          final_t, n_contrib, dimage, slots, bd,
                                                          counter, pc);
      return bwd_go<false, 64, false, false, true, true>(ctx, pb, bb, T, width, height, bg, final_t,
                                                         n_contrib, dimage, slots, bd, counter, pc);
    }
  }
  if (rv.bwd_batch == 16) {
    if (need_abs)
      return bwd_go<true, 16, BATCH, PERSIST, ROWS>(ctx, pb, bb, T, width, height, bg, final_t,
                                                    n_contrib, dimage, slots, bd, counter, pc);
    return bwd_go<false, 16, BATCH, PERSIST, ROWS>(ctx, pb, bb, T, width, height, bg, final_t,
                                                   n_contrib, dimage, slots, bd, counter, pc);
  }
  if (need_abs)
    return bwd_go<true, 32, BATCH, PERSIST, ROWS>(ctx, pb, bb, T, width, height, bg, final_t,
                                                  n_contrib, dimage, slots, bd, counter, pc);
  return bwd_go<false, 32, BATCH, PERSIST, ROWS>(ctx, pb, bb, T, width, height, bg, final_t,
                                                 n_contrib, dimage, slots, bd, counter, pc);
}

template <bool BATCH, bool PERSIST>
void bwd_pick(splat_ctx* ctx, const RasterVariant& rv, const ProjBuffers& pb,
              const BinBuffers& bb, unsigned T, uint32_t width, uint32_t height,
              const float bg[3], const float* final_t, const uint32_t* n_contrib,
              const float* dimage, bool ordered, float* slots, bool need_abs, const BatchDev& bd,
              uint32_t* counter) {
  const unsigned pc = rv.per_cu;
  // the record width (9 or 11 words per entry) follows need_abs in both modes
  if (ordered && need_abs)
    return bwd_ordered_go<true, BATCH, PERSIST>(ctx, pb, bb, T, width, height, bg, final_t,
                                                n_contrib, dimage, slots, bd, counter, pc);
  if (ordered)
    return bwd_ordered_go<false, BATCH, PERSIST>(ctx, pb, bb, T, width, height, bg, final_t,
                                                 n_contrib, dimage, slots, bd, counter, pc);
  if (rv.rows)
    return bwd_rows_pick<BATCH, PERSIST, true>(ctx, rv, pb, bb, T, width, height, bg, final_t,
                                               n_contrib, dimage, slots, need_abs, bd, counter);
  return bwd_rows_pick<BATCH, PERSIST, false>(ctx, rv, pb, bb, T, width, height, bg, final_t,
                                              n_contrib, dimage, slots, need_abs, bd, counter);
}

}  // namespace

void raster_forward_counted(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb,
                            uint32_t width, uint32_t height, const float bg[3], float* image,
                            float* final_t, uint32_t* n_contrib, unsigned long long* pairs) {
  const unsigned T = bb.tiles_x * bb.tiles_y;
  fill_u32(ctx, reinterpret_cast<uint32_t*>(pairs), 2 * kNumPairCounters, 0u);
  launch(ctx, "raster_fwd_count", raster_fwd_kernel<64, false, false, true>, dim3(T), dim3(256),
         0, (const float4*)pb.rec, (const uint32_t*)bb.tile_start, (const uint32_t*)nullptr,
         (const uint32_t*)bb.sorted_gauss, T, bb.tiles_x, width, height, bg[0], bg[1], bg[2],
         image, final_t, n_contrib, BatchDev{}, (uint32_t*)nullptr, pairs);
}

void raster_backward_counted(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb,
                             uint32_t width, uint32_t height, const float bg[3],
                             const float* final_t, const uint32_t* n_contrib,
                             const float* dimage, float* slots, unsigned long long* pairs) {
  const unsigned T = bb.tiles_x * bb.tiles_y;
  launch(ctx, "raster_bwd_count", raster_bwd_kernel<false, 32, false, false, true, true>,
         dim3(T), dim3(256), 0, (const float4*)pb.rec, (const uint32_t*)bb.tile_start,
         (const uint32_t*)nullptr, (const uint32_t*)bb.sorted_gauss,
         (const uint32_t*)bb.sorted_entry, T, bb.tiles_x, width, height, bg[0], bg[1], bg[2],
         (const float*)final_t, (const uint32_t*)n_contrib, dimage, slots, BatchDev{},
         (uint32_t*)nullptr, pairs);
}

void raster_forward(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb, uint32_t width,
                    uint32_t height, const float bg[3], float* image, float* final_t,
                    uint32_t* n_contrib, const RasterVariant& rv, const BatchDev* bd,
                    uint32_t* counter) {
  const unsigned T = bb.tiles_x * bb.tiles_y;
  const BatchDev none{};
  SPLAT_REQUIRE(!rv.persistent || counter, "persistent launch needs a counter");
  if (bd) {
    if (rv.persistent)
      fwd_pick<true, true>(ctx, rv, pb, bb, T, width, height, bg, image, final_t, n_contrib, *bd,
                           counter);
    else
      fwd_pick<true, false>(ctx, rv, pb, bb, T, width, height, bg, image, final_t, n_contrib,
                            *bd, counter);
  } else if (rv.persistent) {
    fwd_pick<false, true>(ctx, rv, pb, bb, T, width, height, bg, image, final_t, n_contrib, none,
                          counter);
  } else {
    fwd_pick<false, false>(ctx, rv, pb, bb, T, width, height, bg, image, final_t, n_contrib,
                           none, counter);
  }
}

void raster_backward(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb, uint32_t width,
                     uint32_t height, const float bg[3], const float* final_t,
                     const uint32_t* n_contrib, const float* dimage, bool ordered, float* slots,
                     bool need_abs, const RasterVariant& rv, const BatchDev* bd,
                     uint32_t* counter) {
  const unsigned T = bb.tiles_x * bb.tiles_y;
  const BatchDev none{};
  SPLAT_REQUIRE(!rv.persistent || counter, "persistent launch needs a counter");
  if (bd) {
    if (rv.persistent)
      bwd_pick<true, true>(ctx, rv, pb, bb, T, width, height, bg, final_t, n_contrib, dimage,
                           ordered, slots, need_abs, *bd, counter);
    else
      bwd_pick<true, false>(ctx, rv, pb, bb, T, width, height, bg, final_t, n_contrib, dimage,
                            ordered, slots, need_abs, *bd, counter);
  } else if (rv.persistent) {
    bwd_pick<false, true>(ctx, rv, pb, bb, T, width, height, bg, final_t, n_contrib, dimage,
                          ordered, slots, need_abs, none, counter);
  } else {
    bwd_pick<false, false>(ctx, rv, pb, bb, T, width, height, bg, final_t, n_contrib, dimage,
                           ordered, slots, need_abs, none, counter);
  }
}

RasterTune tune_raster(splat_ctx* ctx, const ProjBuffers& pb, const BinBuffers& bb,
                       uint32_t width, uint32_t height, const float bg[3], float* image,
                       float* final_t, uint32_t* n_contrib, const float* dimage, bool ordered,
                       float* slots, bool need_abs, const BatchDev* bd, uint32_t* counter) {
  hipEvent_t e0, e1;
  SPLAT_HIP(hipEventCreate(&e0));
  SPLAT_HIP(hipEventCreate(&e1));
  const bool timing = ctx->timing;
  ctx->timing = false;
  RasterTune out;
  try {
    auto time_it = [&](auto&& fn) {
      float best = 1e30f;
      for (int r = 0; r < 3; r++) {
        SPLAT_HIP(hipEventRecord(e0, ctx->stream));
        fn();
        SPLAT_HIP(hipEventRecord(e1, ctx->stream));
        SPLAT_HIP(hipEventSynchronize(e1));
        float ms = 0;
        SPLAT_HIP(hipEventElapsedTime(&ms, e0, e1));
        best = std::min(best, ms);
      }
      return best;
    };
    // the default shape is a candidate of its own where it is not the 64 / 32 entries it means
    // on images with more tiles
    const unsigned T = bb.tiles_x * bb.tiles_y;
    const int def_fwd = !bd && few_fwd(RasterVariant{}, T) ? 0 : 64;
    const int def_bwd = !bd && few_bwd(RasterVariant{}, T) ? 0 : 32;
    out.fwd_ms = out.bwd_ms = 1e30f;
    for (int fb : {0, 32, 64, 128, 256})
      for (int mode = 0; mode < 4; mode++) {
        if (fb == 0 && (def_fwd != 0 || mode > 0)) continue;
        RasterVariant rv;
        rv.fwd_batch = fb;
        rv.persistent = mode > 0;
        rv.per_cu = mode == 1 ? 2 : (mode == 2 ? 4 : 8);
        const float ms = time_it([&] {
          raster_forward(ctx, pb, bb, width, height, bg, image, final_t, n_contrib, rv, bd,
                         counter);
        });
        out.candidates++;
        if (rv.fwd_batch == def_fwd && !rv.persistent) out.default_fwd_ms = ms;
        if (ms < out.fwd_ms) {
          out.fwd_ms = ms;
          out.fwd = rv;
        }
      }
    for (int bw : {0, 16, 32})
      for (int mode = 0; mode < 8; mode++) {
        if (bw == 0 && (ordered || def_bwd != 0 || mode > 0)) continue;
        RasterVariant rv;
        // the ordered form has no such batches and walks per entry: the default is kept
        rv.bwd_batch = ordered ? def_bwd : bw;
        rv.rows = mode < 4 || ordered;
        if (ordered && mode >= 4) continue;
        rv.persistent = mode % 4 > 0;
        rv.per_cu = mode % 4 == 1 ? 2 : (mode % 4 == 2 ? 4 : 8);
        const float ms = time_it([&] {
          raster_backward(ctx, pb, bb, width, height, bg, final_t, n_contrib, dimage, ordered,
                          slots, need_abs, rv, bd, counter);
        });
        out.candidates++;
        if (rv.bwd_batch == def_bwd && !rv.persistent && rv.rows) out.default_bwd_ms = ms;
        if (ms < out.bwd_ms) {
          out.bwd_ms = ms;
          out.bwd = rv;
        }
      }
  } catch (...) {
    ctx->timing = timing;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    throw;
  }
  ctx->timing = timing;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return out;
}

bool supported_batches(const splat_tune_result& shapes) {
  const int f = shapes.fwd_batch, b = shapes.bwd_batch;
  return (f == 0 || f == 32 || f == 64 || f == 128 || f == 256) && (b == 0 || b == 16 || b == 32);
}

void fill_tune_result(const RasterTune& t, splat_tune_result* out) {
  out->fwd_batch = t.fwd.fwd_batch;
  out->fwd_persistent = t.fwd.persistent;
  out->fwd_per_cu = (int32_t)t.fwd.per_cu;
  out->bwd_batch = t.bwd.bwd_batch;
  out->bwd_persistent = t.bwd.persistent;
  out->bwd_per_cu = (int32_t)t.bwd.per_cu;
  out->fwd_ms = t.fwd_ms;
  out->bwd_ms = t.bwd_ms;
  out->default_fwd_ms = t.default_fwd_ms;
  out->default_bwd_ms = t.default_bwd_ms;
  out->candidates = t.candidates;
  out->bwd_row_lists = t.bwd.rows ? 1 : 0;
}

void reduce_slots(splat_ctx* ctx, const uint32_t* entry_offset, const float* slots, size_t n,
                  splat_proj_grad* grads, float* abs_grads, const StepStatus* status) {
  static_assert(sizeof(splat_proj_grad) == 9 * sizeof(float), "slot order of splat_proj_grad");
  if (abs_grads)
    launch(ctx, "reduce_slots", reduce_slots_kernel<11>, dim3(blocks_for(n, 64 / 11)), dim3(64),
           0, entry_offset, slots, (uint32_t)n, grads, abs_grads, status);
  else
    launch(ctx, "reduce_slots", reduce_slots_kernel<9>, dim3(blocks_for(n, 64 / 9)), dim3(64), 0,
           entry_offset, slots, (uint32_t)n, grads, abs_grads, status);
}

}  // namespace splat
