// Learned densification scorer: 12 features -> 64 -> 64 -> 64 (tanh GELU) -> 3 logits
// (clone, split, prune) on the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16: bfloat16
// operands, binary32 accumulation).  No counterpart in the reference, whose densification
// is the threshold heuristic of src/densify.rs:125-221.
//
// Orientation: every layer computes D[unit][sample] = W[unit][in] * X[in][sample] + b, so a
// wave holds 16 samples (the 16 columns of the 16x16 tile) and the output units are the
// rows.  MFMA lane layouts (16x16x32): A: lane l holds row l%16, k = 8(l/16)..+7;
// B: column l%16, k = 8(l/16)..+7; D: column l%16, rows 4(l/16)..+3.  A layer's D values
// become the next layer's B operand without leaving the lane: slot (kb, g = l/16, q) of
// the contraction is taken to be unit h(kb, g, q) = 16(2kb + q/4) + 4g + q%4, exactly the
// units the lane holds, and the weight operands are packed in the same permuted order.
//
// Weight gradients contract over samples, so the error signals and activations of a
// 64-sample chunk are staged in LDS transposed ([unit][sample]) and multiplied there; a
// constant-one input turns the bias gradients into one more output column.
//
// Parameter layout (binary32 master copy): W1[64][12] b1[64] W2[64][64] b2[64] W3[64][64]
// b3[64] W4[3][64] b4[3] (9347 values).
#include "internal.hpp"
#include "mlp.hpp"

namespace splat {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kIn = 12, kHid = 64, kOut = 3;
constexpr int kW1 = 0, kB1 = 768, kW2 = 832, kB2 = 4928, kW3 = 4992, kB3 = 9088, kW4 = 9152,
              kB4 = 9344;
// Packed operand blocks (64 lanes x 8 bfloat16 each): forward A operands of layers 1-4
// (4x1, 4x2, 4x2, 1x2 blocks of M x K), then backward A operands (transposed weights) of
// layers 4, 3, 2 (4x1, 4x2, 4x2).
constexpr int kF1 = 0, kF2 = 4, kF3 = 12, kF4 = 20, kT4 = 22, kT3 = 26, kT2 = 34,
              kBlocks = 42;
constexpr int kChunk = 64;  // samples per workgroup pass of the training kernel
constexpr int kGroups = kChunk / 16;  // samples in groups of 16, one per column of a matrix tile
// bfloat16 values between the LDS rows of two units: 144 bytes, so that the 16 rows which a
// matrix operand is read from, 16 bytes each, lie in different banks
constexpr int kRow = kChunk + 8;
constexpr int kGradThreads = 64 * 4 * kGroups;  // a wave per sample group and M-block

__device__ __forceinline__ __bf16 to_bf16(float x) {  // round to nearest, ties to even
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return __builtin_bit_cast(__bf16, (uint16_t)(u >> 16));
}
__device__ __forceinline__ uint16_t bf16_bits(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// expf_tab without branches, so that a lane's activations interleave: beyond the clamps the
// conversion to binary32 gives its special cases (0 and infinity; NaN passes the compares).
__device__ __forceinline__ float expf_clamp(float x, const uint64_t* tab) {
  const double c0 = 0x1.c6af84b912394p-5 / 32.0 / 32.0 / 32.0;
  const double c1 = 0x1.ebfce50fac4f3p-3 / 32.0 / 32.0;
  const double c2 = 0x1.62e42ff0c52d6p-1 / 32.0;
  const double shift = 0x1.8p+52;
  x = x < -104.0f ? -104.0f : x;
  x = x > 89.0f ? 89.0f : x;
  const double z = 0x1.71547652b82fep+0 * 32.0 * (double)x;
  double kd = z + shift;
  const uint64_t ki = d2bits(kd);
  kd -= shift;
  const double r = z - kd;
  const double s = bits2d(tab[ki % 32] + (ki << 47));
  const double zz = c0 * r + c1;
  const double r2 = r * r;
  double y = c2 * r + 1.0;
  y = zz * r2 + y;
  y = y * s;
  return (float)y;
}

// LDS copy of the table (the barrier is the caller's).
__device__ __forceinline__ void load_exp_table(uint64_t* tab) {
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Table[threadIdx.x];
}

// gelu(z) = 0.5 z (1 + tanh(u)), u = c (z + 0.044715 z^3); also its derivative.
__device__ __forceinline__ float gelu(float z, const uint64_t* tab, float* dg) {
  const float c = 0.7978845608028654f, k = 0.044715f;
  const float u = c * (z + k * z * z * z);
  const float t = 1.0f - 2.0f / (1.0f + expf_clamp(2.0f * u, tab));
  const float du = c * (1.0f + 3.0f * k * z * z);
  *dg = 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * du;
  return 0.5f * z * (1.0f + t);
}

__device__ __forceinline__ bf16x8 blockop(const bf16x8* __restrict__ packed, int block, int lane) {
  return (packed + block * 64)[(uint32_t)lane];  // uniform base, 32-bit lane offset
}

// B operand (slot kb) from the D values of four M-blocks.
__device__ __forceinline__ bf16x8 b_from_d(const f32x4* v, int kb) {
  bf16x8 r;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    r[q] = to_bf16(v[2 * kb][q]);
    r[q + 4] = to_bf16(v[2 * kb + 1][q]);
  }
  return r;
}

// Bias in D layout for M-block mb: rows 16 mb + 4g + r.
__device__ __forceinline__ f32x4 bias_d(const float* __restrict__ b, int nout, int mb, int g) {
  f32x4 c;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int o = 16 * mb + 4 * g + r;
    c[r] = o < nout ? b[o] : 0.0f;
  }
  return c;
}

// Feature operand of one lane: features 8g..8g+7 of its sample (zero beyond 12).
__device__ __forceinline__ bf16x8 feature_operand(const float* f, int g) {
  bf16x8 x;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int k = 8 * g + q;
    x[q] = to_bf16(k < kIn ? f[k] : 0.0f);
  }
  return x;
}

// The same of a layer of kHid units, 16 bytes at a time (kB1 to kB3 are multiples of 4).
__device__ __forceinline__ f32x4 bias4(const float* __restrict__ b, int mb, int g) {
  return *reinterpret_cast<const f32x4*>(b + 16 * mb + 4 * g);
}

// The same pointer, but nothing loaded through it is known to be the same as before: keeps the
// operands and biases of all layers from being hoisted out of a loop into registers.
template <class T>
__device__ __forceinline__ const T* reload(const T* p) {
  asm volatile("" : "+s"(p));
  return p;
}

__device__ __forceinline__ f32x4 gelu4(f32x4 z, const uint64_t* tab, f32x4* d) {
  f32x4 a;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    float dg;
    a[r] = gelu(z[r], tab, &dg);
    (*d)[r] = dg;
  }
  return a;
}

// Logits (D layout, rows 0..2 in lanes 0..15) of a wave's 16 samples.
__device__ __forceinline__ f32x4 forward16(const bf16x8* __restrict__ packed,
                                           const float* __restrict__ p, bf16x8 x, int lane,
                                           const uint64_t* tab) {
  const int g = lane >> 4;
  f32x4 a[4], d;
#pragma unroll
  for (int mb = 0; mb < 4; mb++)
    a[mb] = gelu4(mfma(blockop(packed, kF1 + mb, lane), x, bias4(p + kB1, mb, g)), tab, &d);
#pragma unroll
  for (int layer = 2; layer <= 3; layer++) {
    const int f = layer == 2 ? kF2 : kF3, bias = layer == 2 ? kB2 : kB3;
    const bf16x8 b0 = b_from_d(a, 0), b1 = b_from_d(a, 1);
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
      f32x4 z = bias4(p + bias, mb, g);
      z = mfma(blockop(packed, f + 2 * mb, lane), b0, z);
      a[mb] = gelu4(mfma(blockop(packed, f + 2 * mb + 1, lane), b1, z), tab, &d);
    }
  }
  f32x4 z = bias_d(p + kB4, kOut, 0, g);
  z = mfma(blockop(packed, kF4, lane), b_from_d(a, 0), z);
  return mfma(blockop(packed, kF4 + 1, lane), b_from_d(a, 1), z);
}

// Packs the binary32 master weights into the bfloat16 operand blocks.
__global__ void __launch_bounds__(256) mlp_pack_kernel(const float* __restrict__ p,
                                                       bf16x8* __restrict__ packed) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;  // one lane of one block
  if (t >= kBlocks * 64) return;
  const int block = t / 64, lane = t % 64, g = lane >> 4, row16 = lane & 15;
  bf16x8 out;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    float v = 0.0f;
    const int hperm = 4 * g + (q & 3);  // + 16 (2 kb + q / 4)
    if (block < kF2) {  // layer 1 forward: K = features in natural order
      const int o = 16 * block + row16, k = 8 * g + q;
      v = k < kIn ? p[kW1 + o * kIn + k] : 0.0f;
    } else if (block < kT4) {  // layers 2-4 forward
      int L, mb, kb;
      if (block < kF3) {
        L = 2, mb = (block - kF2) / 2, kb = (block - kF2) % 2;
      } else if (block < kF4) {
        L = 3, mb = (block - kF3) / 2, kb = (block - kF3) % 2;
      } else {
        L = 4, mb = 0, kb = block - kF4;
      }
      const int o = 16 * mb + row16, h = 16 * (2 * kb + q / 4) + hperm;
      const int nout = L == 4 ? kOut : kHid;
      const int base = L == 2 ? kW2 : (L == 3 ? kW3 : kW4);
      v = o < nout ? p[base + o * kHid + h] : 0.0f;
    } else {  // backward: transposed weights, rows = input units of layer L
      int L, mb, kb;
      if (block < kT3) {
        L = 4, mb = block - kT4, kb = 0;
      } else if (block < kT2) {
        L = 3, mb = (block - kT3) / 2, kb = (block - kT3) % 2;
      } else {
        L = 2, mb = (block - kT2) / 2, kb = (block - kT2) % 2;
      }
      const int i = 16 * mb + row16, h = 16 * (2 * kb + q / 4) + hperm;
      const int nout = L == 4 ? kOut : kHid;
      const int base = L == 2 ? kW2 : (L == 3 ? kW3 : kW4);
      v = h < nout ? p[base + h * kHid + i] : 0.0f;
    }
    out[q] = to_bf16(v);
  }
  packed[t] = out;
}

// Logits of n feature rows ([n][12] -> [n][3]); one wave per 16 samples, grid-stride.  Bound by
// the vector instructions of the activations: 93 us at 300k rows (135 us with branches in the
// exponential and all operands held in registers).
__global__ void __launch_bounds__(256) mlp_forward_kernel(const bf16x8* __restrict__ packed,
                                                          const float* __restrict__ p,
                                                          const float* __restrict__ feats,
                                                          uint32_t n, float* __restrict__ logits) {
  __shared__ uint64_t tab[32];
  load_exp_table(tab);
  __syncthreads();
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const uint32_t waves = gridDim.x * (blockDim.x / 64);
  const uint32_t wave = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  for (uint32_t base = wave * 16; base < n; base += waves * 16) {
    const uint32_t s = base + (lane & 15);
    float f[kIn];
#pragma unroll
    for (int k = 0; k < kIn; k++) f[k] = s < n ? feats[(size_t)s * kIn + k] : 0.0f;
    const f32x4 z = forward16(reload(packed), reload(p), feature_operand(f, g), lane, tab);
    if (g == 0 && s < n) {
#pragma unroll
      for (int o = 0; o < kOut; o++) logits[(size_t)s * kOut + o] = z[o];
    }
  }
}

__device__ __forceinline__ float softplus(float z) {
  return z > 0.0f ? z + log1pf(splat_expf(-z)) : log1pf(splat_expf(z));
}

// bfloat16 D values of one M-block, as half a B operand of the next layer: units
// 16 mb + 4g .. + 3 of the lane's sample.
__device__ __forceinline__ uint2 pack4(f32x4 v) {
  return make_uint2(bf16_bits(v[0]) | (uint32_t)bf16_bits(v[1]) << 16,
                    bf16_bits(v[2]) | (uint32_t)bf16_bits(v[3]) << 16);
}

// Stage one M-block of one wave's 16 samples (D layout, packed) into an LDS [unit][sample] array.
__device__ __forceinline__ void stage(uint16_t* s, uint2 v, int mb, int lane, int group) {
  uint16_t* at = s + (16 * mb + 4 * (lane >> 4)) * kRow + 16 * group + (lane & 15);
  at[0] = (uint16_t)v.x;
  at[kRow] = (uint16_t)(v.x >> 16);
  at[2 * kRow] = (uint16_t)v.y;
  at[3 * kRow] = (uint16_t)(v.y >> 16);
}

// The operand of 16 units over staged samples 32 kb .. 32 kb + 31.
__device__ __forceinline__ bf16x8 staged(const uint16_t* s, int mb, int kb, int lane) {
  return *reinterpret_cast<const bf16x8*>(s + (16 * mb + (lane & 15)) * kRow + 32 * kb +
                                          8 * (lane >> 4));
}

// Write a 16x16 tile of weight gradients (row block mb, column block nb; `nin` columns are
// inputs, the next is the bias) to its places in a gradient row.
__device__ __forceinline__ void write_tile(float* __restrict__ row, int wbase, int bbase, int nin,
                                           int nout, int mb, int nb, int lane, f32x4 v) {
  const int in = 16 * nb + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int out = 16 * mb + 4 * (lane >> 4) + r;
    if (out >= nout) continue;
    if (in < nin)
      row[wbase + out * nin + in] = v[r];
    else if (in == nin)
      row[bbase + out] = v[r];
  }
}

// Gradient of the weighted binary cross-entropy over `count` samples (ids order[0..count)
// or 0..count), scaled by inv_batch.  Each workgroup accumulates its chunks' weight
// gradients in registers and writes one partial gradient row (kMlpParams floats) plus its
// partial loss; mlp_adam_kernel sums the rows in workgroup order.
//
// Wave w has sample group w % 4 (16 samples) and M-block w / 4 (16 units) of every hidden layer:
// a layer's values are exchanged through LDS, where the weight gradients find them too.  Of
// those, the waves of M-block mb take layers 3 and 2's row block mb (groups 0 and 1 layer 3's
// columns, 2 and 3 layer 2's), layer 1's (group 1) and layer 4's column block mb (group 3).
// Every tile is summed over a chunk's 64 samples in one accumulator and over the rows in
// order.  Bound by the chain of seven layers, mostly the vector instructions of the
// activations: a wave has 12 per lane, four waves share a SIMD.  A batch of 4096 makes 64
// workgroups, 20.7 us; workgroups of four waves with 48 activations per lane took 22.5 us, and
// 31.7 us with two barriers per layer and LDS rows of 128 bytes, all in the same banks.  (128
// workgroups of 32 samples took 15.2 us, but sum each weight gradient in other parts.)
__global__ void __launch_bounds__(kGradThreads) mlp_grad_kernel(
    const bf16x8* __restrict__ packed, const float* __restrict__ p,
    const float* __restrict__ feats, const uint8_t* __restrict__ labels,
    const float* __restrict__ weights, const uint32_t* __restrict__ order, uint32_t count,
    float inv_batch, float* __restrict__ partial, float* __restrict__ partial_loss) {
  // errors of layers 4 to 1, activations 3 to 1 and features
  __shared__ __attribute__((aligned(16))) uint16_t sE4[16 * kRow], sE3[64 * kRow],
      sE2[64 * kRow], sE1[64 * kRow], sA3[64 * kRow], sA2[64 * kRow], sA1[64 * kRow],
      sX[16 * kRow];
  __shared__ uint2 exch[5][kGroups][4][64];  // activations 1 to 3, errors 3 and 2; group, M-block, lane
  __shared__ float sloss[kGroups];
  __shared__ uint64_t tab[32];
  load_exp_table(tab);
  __syncthreads();
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave % kGroups, mb = wave / kGroups;
  // columns of layer 3 (groups 0, 1) or 2: blocks 0 to 2 (even groups) or block 3 and the bias;
  // then layer 1 (group 1) or layer 4 and its bias (group 3)
  f32x4 acc[4];
#pragma unroll
  for (int k = 0; k < 4; k++) acc[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const __bf16 one = (lane & 15) == 0 ? __builtin_bit_cast(__bf16, (uint16_t)0x3F80)
                                      : __builtin_bit_cast(__bf16, (uint16_t)0);
  const bf16x8 ones = {one, one, one, one, one, one, one, one};  // the constant-one input
  // hand a layer's values on: the whole group's as the next layer's two B operands
  const auto exchange = [&](int slot, uint2 v, bf16x8* b0, bf16x8* b1) {
    exch[slot][group][mb][lane] = v;
    __syncthreads();
    const uint2 u0 = exch[slot][group][0][lane], u1 = exch[slot][group][1][lane],
                u2 = exch[slot][group][2][lane], u3 = exch[slot][group][3][lane];
    *b0 = __builtin_bit_cast(bf16x8, make_uint4(u0.x, u0.y, u1.x, u1.y));
    *b1 = __builtin_bit_cast(bf16x8, make_uint4(u2.x, u2.y, u3.x, u3.y));
  };
  float lsum = 0.0f;
  const uint32_t chunks = (count + kChunk - 1) / kChunk;
  for (uint32_t ch = blockIdx.x; ch < chunks; ch += gridDim.x) {
    const uint32_t idx = ch * kChunk + 16 * group + (lane & 15);
    const bool valid = idx < count;
    const uint32_t s = valid ? (order ? order[idx] : idx) : 0;
    float f[kIn];
#pragma unroll
    for (int k = 0; k < kIn; k++) f[k] = valid ? feats[(size_t)s * kIn + k] : 0.0f;
    const float w = valid ? weights[s] : 0.0f;
    const uint32_t y = valid ? labels[s] : 0u;
    const f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
    if (mb == 0 && g < 2) {
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int k = 8 * g + q;
        const float x = k < kIn ? f[k] : 0.0f;
        sX[k * kRow + 16 * group + (lane & 15)] = k == kIn ? 0x3F80 : bf16_bits(x);
      }
    }
    // A layer's operands and bias are loaded no earlier than beside the layer before it: all
    // layers' would not fit the 128 registers of a lane.
    const bf16x8* at = packed;
    const float* bias = p;
    const auto next_layer = [&] {
      at = reload(at);
      bias = reload(bias);
    };
    next_layer();
    f32x4 d1, d2, d3;
    bf16x8 b0, b1;
    f32x4 z = mfma(blockop(at, kF1 + mb, lane), feature_operand(f, g), bias4(bias + kB1, mb, g));
    next_layer();
    uint2 v = pack4(gelu4(z, tab, &d1));
    stage(sA1, v, mb, lane, group);
    exchange(0, v, &b0, &b1);
    z = mfma(blockop(at, kF2 + 2 * mb, lane), b0, bias4(bias + kB2, mb, g));
    z = mfma(blockop(at, kF2 + 2 * mb + 1, lane), b1, z);
    next_layer();
    v = pack4(gelu4(z, tab, &d2));
    stage(sA2, v, mb, lane, group);
    exchange(1, v, &b0, &b1);
    z = mfma(blockop(at, kF3 + 2 * mb, lane), b0, bias4(bias + kB3, mb, g));
    z = mfma(blockop(at, kF3 + 2 * mb + 1, lane), b1, z);
    next_layer();
    v = pack4(gelu4(z, tab, &d3));
    stage(sA3, v, mb, lane, group);
    exchange(2, v, &b0, &b1);
    z = mfma(blockop(at, kF4, lane), b0, bias_d(bias + kB4, kOut, 0, g));
    z = mfma(blockop(at, kF4 + 1, lane), b1, z);
    next_layer();
    // output error (rows 0..2 live in lanes g == 0), on each of the group's waves
    f32x4 e4 = none;
    if (g == 0 && valid) {
#pragma unroll
      for (int o = 0; o < kOut; o++) {
        const float yo = (y >> o) & 1u ? 1.0f : 0.0f;
        if (mb == 0) lsum += w * (softplus(z[o]) - yo * z[o]) * inv_batch;
        const float sg = 1.0f / (1.0f + expf_clamp(-z[o], tab));
        e4[o] = w * (sg - yo) * inv_batch;
      }
    }
    v = pack4(e4);
    if (mb == 0) stage(sE4, v, 0, lane, group);
    const bf16x8 E = __builtin_bit_cast(bf16x8, make_uint4(v.x, v.y, 0u, 0u));
    v = pack4(mfma(blockop(at, kT4 + mb, lane), E, none) * d3);
    stage(sE3, v, mb, lane, group);
    exchange(3, v, &b0, &b1);
    z = mfma(blockop(at, kT3 + 2 * mb, lane), b0, none);
    v = pack4(mfma(blockop(at, kT3 + 2 * mb + 1, lane), b1, z) * d2);
    stage(sE2, v, mb, lane, group);
    exchange(4, v, &b0, &b1);
    z = mfma(blockop(at, kT2 + 2 * mb, lane), b0, none);
    v = pack4(mfma(blockop(at, kT2 + 2 * mb + 1, lane), b1, z) * d1);
    stage(sE1, v, mb, lane, group);
    __syncthreads();
    const uint16_t *se = group < 2 ? sE3 : sE2, *sa = group < 2 ? sA2 : sA1;
#pragma unroll
    for (int kb = 0; kb < kChunk / 32; kb++) {
      const bf16x8 e = staged(se, mb, kb, lane);
      if (group % 2 == 0) {
#pragma unroll
        for (int nb = 0; nb < 3; nb++) acc[nb] = mfma(e, staged(sa, nb, kb, lane), acc[nb]);
      } else {
        acc[0] = mfma(e, staged(sa, 3, kb, lane), acc[0]);
        acc[1] = mfma(e, ones, acc[1]);
      }
      if (group == 1) {
        acc[2] = mfma(staged(sE1, mb, kb, lane), staged(sX, 0, kb, lane), acc[2]);
      } else if (group == 3) {
        const bf16x8 e4b = staged(sE4, 0, kb, lane);
        acc[2] = mfma(e4b, staged(sA3, mb, kb, lane), acc[2]);
        acc[3] = mfma(e4b, ones, acc[3]);
      }
    }
    __syncthreads();
  }
  // write this workgroup's gradient row
  float* row = partial + (size_t)blockIdx.x * kMlpParams;
  const int wbase = group < 2 ? kW3 : kW2, bbase = group < 2 ? kB3 : kB2;
  if (group % 2 == 0) {
#pragma unroll
    for (int nb = 0; nb < 3; nb++) write_tile(row, wbase, bbase, kHid, kHid, mb, nb, lane, acc[nb]);
  } else {
    write_tile(row, wbase, bbase, kHid, kHid, mb, 3, lane, acc[0]);
    write_tile(row, wbase, bbase, kHid, kHid, mb, 4, lane, acc[1]);
  }
  if (group == 1) {
    write_tile(row, kW1, kB1, kIn, kHid, mb, 0, lane, acc[2]);
  } else if (group == 3) {
    write_tile(row, kW4, kB4, kHid, kOut, 0, mb, lane, acc[2]);
    if (mb == 0) write_tile(row, kW4, kB4, kHid, kOut, 0, 4, lane, acc[3]);
  }
  if (mb == 0) {
    for (int d = 32; d >= 1; d >>= 1) lsum += __shfl_xor(lsum, d, 64);
    if (lane == 0) sloss[group] = lsum;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    partial_loss[blockIdx.x] = ((sloss[0] + sloss[1]) + sloss[2]) + sloss[3];
}

// Parameter k's places among the packed operands (the inverse of mlp_pack_kernel's map).
__device__ __forceinline__ void pack_one(uint16_t* __restrict__ packed, int k, float value) {
  const uint16_t b = bf16_bits(value);
  const auto put = [&](int block, int lane, int q) { packed[(block * 64 + lane) * 8 + q] = b; };
  const auto slot = [&](int block, int row16, int h) {  // of row row16, hidden unit h
    put(block + h / 32, 16 * (h % 16 / 4) + row16, 4 * (h / 16 % 2) + h % 4);
  };
  if (k < kB1) {
    const int o = k / kIn, i = k % kIn;
    put(kF1 + o / 16, 16 * (i / 8) + o % 16, i % 8);
  } else if (k >= kW2 && k < kB2) {
    const int o = (k - kW2) / kHid, i = (k - kW2) % kHid;
    slot(kF2 + 2 * (o / 16), o % 16, i);
    slot(kT2 + 2 * (i / 16), i % 16, o);
  } else if (k >= kW3 && k < kB3) {
    const int o = (k - kW3) / kHid, i = (k - kW3) % kHid;
    slot(kF3 + 2 * (o / 16), o % 16, i);
    slot(kT3 + 2 * (i / 16), i % 16, o);
  } else if (k >= kW4 && k < kB4) {
    const int o = (k - kW4) / kHid, i = (k - kW4) % kHid;
    slot(kF4, o, i);
    slot(kT4 + i / 16, i % 16, o);
  }
}

constexpr int kAdamThreads = 64;
constexpr int kAdamRows = 16;  // rows in flight per lane

// Sums the workgroups' gradient rows in order; optionally writes the gradient and/or
// applies Adam to the master weights, whose packed operands (all zero where they hold no
// weight) it rewrites.  The last workgroup sums the partial losses in order.  Bound by the
// latency of the row loads: a wave per workgroup and 16 rows in flight instead of 256 lanes and
// the few rows of the compiler's own unrolling, 5.2 us at 64 rows (16.6 us, and 9.9 us for the
// losses and operands as launches of their own).
__global__ void __launch_bounds__(kAdamThreads) mlp_adam_kernel(
    float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
    uint16_t* __restrict__ packed, const float* __restrict__ partial,
    const float* __restrict__ partial_loss, uint32_t rows, float* __restrict__ grad_out,
    float* __restrict__ loss_out, int update, float lr, float c1, float c2) {
  if (blockIdx.x == gridDim.x - 1) {
    float s = 0.0f;
    for (uint32_t r0 = 0; r0 < rows; r0 += 64) {
      const uint32_t r = r0 + threadIdx.x;
      const float x = r < rows ? partial_loss[r] : 0.0f;
      const uint32_t cnt = min(64u, rows - r0);
      for (uint32_t k = 0; k < cnt; k++)
        s += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), (int)k));
    }
    if (threadIdx.x == 0) *loss_out = s;
    return;
  }
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (uint32_t)kMlpParams) return;
  const float* at = partial + k;
  float gsum = 0.0f;
  uint32_t r = 0;
  for (; r + kAdamRows <= rows; r += kAdamRows, at += (size_t)kAdamRows * kMlpParams) {
    float x[kAdamRows];
#pragma unroll
    for (int q = 0; q < kAdamRows; q++) x[q] = at[(size_t)q * kMlpParams];
#pragma unroll
    for (int q = 0; q < kAdamRows; q++) gsum += x[q];
  }
  for (; r < rows; r++, at += kMlpParams) gsum += *at;
  if (grad_out) grad_out[k] = gsum;
  if (!update) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  m[k] = b1 * m[k] + (1.0f - b1) * gsum;
  v[k] = b2 * v[k] + (1.0f - b2) * gsum * gsum;
  const float w = p[k] - lr * (m[k] / c1) / (sqrtf(v[k] / c2) + eps);
  p[k] = w;
  pack_one(packed, (int)k, w);
}

}  // namespace

size_t mlp_packed_bytes() { return (size_t)kBlocks * 64 * 16; }

void mlp_pack(splat_ctx* ctx, const float* params, void* packed) {
  launch(ctx, "mlp_pack", mlp_pack_kernel, dim3(blocks_for(kBlocks * 64, 256)), dim3(256), 0,
         params, (bf16x8*)packed);
}

void mlp_forward(splat_ctx* ctx, const void* packed, const float* params, const float* feats,
                 size_t n, float* logits) {
  const unsigned blocks = std::min<unsigned>(blocks_for(n, 64), 4096u);
  launch(ctx, "mlp_forward", mlp_forward_kernel, dim3(blocks), dim3(256), 0,
         (const bf16x8*)packed, params, feats, (uint32_t)n, logits);
}

unsigned mlp_grad_rows(size_t count) {
  return std::max<unsigned>(1u, std::min<unsigned>(blocks_for(count, kChunk), 256u));
}

void mlp_grad(splat_ctx* ctx, const void* packed, const float* params, const float* feats,
              const uint8_t* labels, const float* weights, const uint32_t* order, size_t count,
              float inv_batch, float* partial, float* partial_loss) {
  launch(ctx, "mlp_grad", mlp_grad_kernel, dim3(mlp_grad_rows(count)), dim3(kGradThreads), 0,
         (const bf16x8*)packed, params, feats, labels, weights, order, (uint32_t)count,
         inv_batch, partial, partial_loss);
}

void mlp_reduce_update(splat_ctx* ctx, float* params, float* m, float* v, void* packed,
                       const float* partial, const float* partial_loss, unsigned rows,
                       float* grad_out, float* loss_out, bool update, float lr, float c1,
                       float c2) {
  launch(ctx, "mlp_adam", mlp_adam_kernel, dim3(blocks_for(kMlpParams, kAdamThreads) + 1),
         dim3(kAdamThreads), 0, params, m, v, (uint16_t*)packed, partial, partial_loss, rows,
         grad_out, loss_out, update ? 1 : 0, lr, c1, c2);
}

}  // namespace splat
