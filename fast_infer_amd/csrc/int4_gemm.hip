// INT4 group-quantized linear layers for gfx950: quantize, dequantize, and C = X * W^T
// with the dequantization fused into the MFMA loop.
//
// Wire format (loader.py:9-41): W [N, K] is stored as int8 bytes [N, K/2]; byte j of a
// row holds k = 2j in its low nibble and k = 2j+1 in its high nibble, each a 4-bit two's
// complement value in [-8, 7]; scales are fp16 [N, K/128], one per 128-wide group.
// The weight the reference multiplies with is fp16(q * scale) (matmul.py:83-84 and
// :309-326): one rounding of an exact product, which is what v_pk_mul_f16 computes.
//
// C[m, n] = fp16( sum_k X[m, k] * W[n, k] ), fp32 accumulation (matmul.py:14-132,
// :135-186).  By the rows M of X and the measured costs in plan():
//   up to 16 rows where it is the fastest, and up to 4 with a fused norm:
//                     gemv_kernel: one workgroup per 16 output columns, K split over its waves;
//   packed weights:   mid_gemm_kernel, which unpacks them in registers, and for many row tiles
//                     one unpacking into the workspace followed by tile_gemm_kernel;
//   fp16 weights:     tile_gemm_kernel.
// The last two split K over workgroups where the tiles alone leave CUs idle, and add the splits
// inside the launch (add_splits).  gemm_kernel serves rows of X too far apart for their 32-bit
// offsets: one workgroup = 4 waves = 64 output columns (16 per wave) x MT rows, X[MT, 128] per
// group staged through registers in LDS (double buffered, rows padded to 272 bytes so the 16
// rows a wave reads are on distinct banks), K split over blockIdx.z.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace fi {
namespace gemm {

constexpr int kThreads = 256;
constexpr int kNTile = 64;
constexpr int kGroup = 128;     // K per scale group and per pipeline step
constexpr int kLdsRow = 136;    // halves per staged X row (128 + 8 pad)
constexpr int kFusedNormM = 4;  // rows up to which gemv_kernel takes the RMSNorm in

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

struct Params {
  const half_t* x;
  int64_t x_stride;  // elements between rows of X
  int M, K, N;
  const uint8_t* w;  // int4 bytes [N, K/2] or fp16 [N, K]
  int64_t w_stride;  // bytes (int4) or elements (fp16) between rows of W
  const half_t* scales;
  int64_t s_stride;  // elements between rows of scales
  half_t* out;
  int64_t out_stride;
  float* partial;    // [splits, M, N] fp32 when splits > 1
  int groups_per_split;
  const half_t* norm_w;  // RMSNorm weight [K] when the norm is fused into the X operand
  float eps;
  // mid_gemm_kernel and tile_gemm_kernel: row tiles, all tiles, K splits, the per-tile arrival
  // counters (one line set per XCD group, counter_stride apart); row tiles per XCD when they
  // are banded (tile_gemm_kernel), else 0; 16-byte output stores
  int tiles_m;
  int tiles;
  int ksplit;
  unsigned* counters;
  int counter_stride;
  int band;
  int vec_out;
};

__device__ __forceinline__ uint32_t as_u32(half2_t h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ half2_t as_h2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }

// Eight int4 values (natural k order, nibble i = k0 + i) -> fp16(q * s).
//
// With e = d >> 4, byte j of e holds nibble 2j + 1 in its low half.  Two byte
// permutations put byte j of d beside byte j of e, so that the low nibbles at bits 0 and
// 16 are the k pairs (0, 1) and (4, 5), and 8 bits higher (2, 3) and (6, 7): every pair
// comes out in MFMA order, with no permutation after the arithmetic (22 VALU instructions as
// compiled: each mask-and-insert is a v_and_b32 + v_or_b32 pair).
__device__ __forceinline__ half8 dequant8(uint32_t d, half2_t s2) {
#pragma clang fp contract(off)
  d ^= 0x88888888u;  // two's complement nibble n -> n + 8 in [0, 15]
  const uint32_t e = d >> 4;
  const uint32_t lo = __builtin_amdgcn_perm(e, d, 0x05040100u);  // d.b0 d.b1 e.b0 e.b1
  const uint32_t hi = __builtin_amdgcn_perm(e, d, 0x07060302u);  // d.b2 d.b3 e.b2 e.b3
  // 0x6400 | v is the fp16 value 1024 + v; minus 1032 gives the signed nibble exactly
  const half2_t bias = {(half_t)1032.0f, (half_t)1032.0f};
  u32x4 r;
  r[0] = as_u32((as_h2((lo & 0x000F000Fu) | 0x64006400u) - bias) * s2);         // k0, k1
  r[1] = as_u32((as_h2(((lo >> 8) & 0x000F000Fu) | 0x64006400u) - bias) * s2);  // k2, k3
  r[2] = as_u32((as_h2((hi & 0x000F000Fu) | 0x64006400u) - bias) * s2);         // k4, k5
  r[3] = as_u32((as_h2(((hi >> 8) & 0x000F000Fu) | 0x64006400u) - bias) * s2);  // k6, k7
  return as_half8(r);
}

// Store C[m][nb .. nb + 3] (columns past N dropped): to the fp32 partials of split
// blockIdx.z, or as fp16 to the output.
__device__ __forceinline__ void store_row_piece(const Params& p, floatx4 v, int m, int nb) {
  if (p.partial) {
    float* dst = p.partial + ((int64_t)blockIdx.z * p.M + m) * p.N + nb;
    if (nb + 3 < p.N && (p.N & 3) == 0) {
      *(floatx4*)dst = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nb + i < p.N) dst[i] = v[i];
    }
  } else {
    half_t* dst = p.out + (int64_t)m * p.out_stride + nb;
    const half4 h = to_half4(v);
    if (nb + 3 < p.N && ((uintptr_t)dst & 7) == 0) {
      *(half4*)dst = h;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nb + i < p.N) dst[i] = h[i];
    }
  }
}

// Store a workgroup's 64-column x (16 * kMSub)-row tile.  Lane (row, grp) of wave w holds
// C[m0 + 16j + row][n0 + 16w + 4grp + i] in acc[j][i].  With K split over blockIdx.z the
// tile goes to the fp32 partials (reduce_kernel adds them), otherwise to the fp16 output.
template <int kMSub>
__device__ __forceinline__ void store_tile(const Params& p, const floatx4 (&acc)[kMSub], int m0,
                                           int n0) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row = lane & 15;
  const int nb = n0 + wave * 16 + 4 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < kMSub; ++j) {
    const int m = m0 + 16 * j + row;
    if (m < p.M) store_row_piece(p, acc[j], m, nb);
  }
}

// ---------------------------------------------------------------------------------------
// RMSNorm (kernels/rms_norm.py:8-43): y = fp16((x * r) * w) with r = rsqrt(sum(x^2)/K + eps),
// all in fp32.  One wave reduces one row.

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Rows up to kRowChunks * 512 elements are held in registers (16 bytes per lane per 512
// elements), every load issued before the first use; longer rows loop.
constexpr int kRowChunks = 16;

__device__ __forceinline__ float sum_sq8(u32x4 v) {
  const half8 h = as_half8(v);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s += (float)h[e] * (float)h[e];
  return s;
}

// r of one row of K (a multiple of 8) elements, computed by the calling wave
__device__ __forceinline__ float row_rsqrt(const half_t* xrow, int K, float eps, int lane) {
  float s = 0.f;
  if (K <= kRowChunks * 512) {
    u32x4 v[kRowChunks];
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) {
      const int k = lane * 8 + i * 512;
      v[i] = k < K ? *(const u32x4*)(xrow + k) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) s += sum_sq8(v[i]);
  } else {
    for (int k = lane * 8; k < K; k += 512) s += sum_sq8(*(const u32x4*)(xrow + k));
  }
  s = wave_sum(s);
  return rsqrtf(s / (float)K + eps);
}

// eight normalized elements: fp16((x * r) * w), products rounded separately (no fma)
__device__ __forceinline__ u32x4 norm8(u32x4 xv, float r, u32x4 wv) {
#pragma clang fp contract(off)
  const half8 x = as_half8(xv);
  const half8 w = as_half8(wv);
  half8 y;
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = (half_t)(((float)x[e] * r) * (float)w[e]);
  return as_u32x4(y);
}

__global__ __launch_bounds__(256) void rmsnorm_kernel(const half_t* x, int64_t x_stride, int M,
                                                      int K, const half_t* w, float eps,
                                                      half_t* out, int64_t out_stride) {
  const int lane = threadIdx.x & 63;
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  const half_t* xr = x + (int64_t)m * x_stride;
  half_t* o = out + (int64_t)m * out_stride;
  if (K <= kRowChunks * 512) {  // the row is read once, into registers
    u32x4 v[kRowChunks], wv[kRowChunks];
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) {
      const int k = lane * 8 + i * 512;
      v[i] = k < K ? *(const u32x4*)(xr + k) : u32x4{0, 0, 0, 0};
      wv[i] = k < K ? *(const u32x4*)(w + k) : u32x4{0, 0, 0, 0};
    }
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) s += sum_sq8(v[i]);
    const float r = rsqrtf(wave_sum(s) / (float)K + eps);
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) {
      const int k = lane * 8 + i * 512;
      if (k < K) *(u32x4*)(o + k) = norm8(v[i], r, wv[i]);
    }
    return;
  }
  const float r = row_rsqrt(xr, K, eps, lane);
  for (int k = lane * 8; k < K; k += 512)
    *(u32x4*)(o + k) = norm8(*(const u32x4*)(xr + k), r, *(const u32x4*)(w + k));
}

// rmsnorm_kernel with a workgroup per row (K up to 8192): every thread takes a few elements, the
// waves' sums of squares meet in LDS.  A wave per row left few rows on a quarter of the
// workgroups and loaded its 16 chunks one guarded load after another: rows of 3072 elements
// 5.0 -> 3.4 us for 64 rows, 5.8 -> 5.1 for 1000, 37.5 -> 35.6 (5.7 TB/s) for 16384; of 8192 7.6 ->
// 3.8 for 64.  Rows of up to 2048 elements leave threads idle, which many of them notice: 768
// elements 4.5 -> 4.2 us for 1000 rows, but 17.3 against 21.2 for 16384, so they stay with
// rmsnorm_kernel from kWaveRows rows; those of less than 2816, whose second part leaves three of
// four waves idle, from kMoreRows (2056 elements, 12288 rows 19.9 against 18.4, 16384 28.4 against
// 32.6; 2560 elements, 16384 rows 32.0 against 33.0); and all from kManyRows, whose 256 threads a
// row are more than a launch takes (2^32 along x).
constexpr int kRowParts = 4;
constexpr int kWaveRows = 1024;
constexpr int kMoreRows = 13000;
constexpr int64_t kManyRows = 1 << 24;
__global__ __launch_bounds__(256) void rmsnorm_row_kernel(const half_t* x, int64_t x_stride, int K,
                                                          const half_t* w, float eps, half_t* out,
                                                          int64_t out_stride) {
  __shared__ float part[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // elements past K read zeros through the buffer bounds
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(x + (int64_t)blockIdx.x * x_stride), (short)0, K * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, K * 2, 0x00020000);
  u32x4 v[kRowParts], wv[kRowParts];
#pragma unroll
  for (int i = 0; i < kRowParts; ++i) {
    const int k2 = (threadIdx.x * 8 + i * 2048) * 2;
    v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, k2, 0, 0));
    wv[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, k2, 0, 0));
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kRowParts; ++i) s += sum_sq8(v[i]);
  s = wave_sum(s);
  if (lane == 0) part[wave] = s;
  __syncthreads();
  const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / (float)K + eps);
  half_t* o = out + (int64_t)blockIdx.x * out_stride;
#pragma unroll
  for (int i = 0; i < kRowParts; ++i) {
    const int k = threadIdx.x * 8 + i * 2048;
    if (k < K) *(u32x4*)(o + k) = norm8(v[i], r, wv[i]);
  }
}

// One row normalized by the calling wave into dst (LDS or global), K a multiple of 8.
__device__ __forceinline__ void norm_row_to(const half_t* xr, const half_t* w, int K, float eps,
                                            half_t* dst, int lane) {
  if (K <= kRowChunks * 512) {
    u32x4 v[kRowChunks];
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) {
      const int k = lane * 8 + i * 512;
      v[i] = k < K ? *(const u32x4*)(xr + k) : u32x4{0, 0, 0, 0};
    }
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) s += sum_sq8(v[i]);
    const float r = rsqrtf(wave_sum(s) / (float)K + eps);
#pragma unroll
    for (int i = 0; i < kRowChunks; ++i) {
      const int k = lane * 8 + i * 512;
      if (k < K) *(u32x4*)(dst + k) = norm8(v[i], r, *(const u32x4*)(w + k));
    }
    return;
  }
  const float r = row_rsqrt(xr, K, eps, lane);
  for (int k = lane * 8; k < K; k += 512)
    *(u32x4*)(dst + k) = norm8(*(const u32x4*)(xr + k), r, *(const u32x4*)(w + k));
}

template <int MT, bool kInt4>
__global__ __launch_bounds__(kThreads, 2) void gemm_kernel(Params p) {
  constexpr int kMSub = MT / 16;          // 16-row MFMA tiles per wave
  constexpr int kXLoads = MT / 16;        // 16-byte X loads per thread per group
  __shared__ __attribute__((aligned(16))) half_t xs[2][MT * kLdsRow];

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row = lane & 15;
  const int grp = lane >> 4;
  const int n = blockIdx.x * kNTile + wave * 16 + row;  // this lane's weight row
  const int nc = n < p.N ? n : p.N - 1;                 // rows past N compute, never store
  const int m0 = blockIdx.y * MT;
  const int groups = p.K / kGroup;
  const int g_begin = blockIdx.z * p.groups_per_split;
  const int g_end = min(g_begin + p.groups_per_split, groups);

  // X staging: thread t moves 16 bytes of rows t/16 + 16i, chunk t%16
  const int xr = threadIdx.x >> 4;
  const int xc = threadIdx.x & 15;
  u32x4 xreg[kXLoads];
  auto load_x = [&](int g) {
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) {
      const int m = m0 + xr + 16 * i;
      if (m < p.M)
        xreg[i] = *(const u32x4*)(p.x + (int64_t)m * p.x_stride + g * kGroup + xc * 8);
      else
        xreg[i] = u32x4{0, 0, 0, 0};
    }
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kXLoads; ++i)
      *(u32x4*)(&xs[buf][(xr + 16 * i) * kLdsRow + xc * 8]) = xreg[i];
  };

  // weights of this lane for one group: 16 bytes (int4) or 4 x 16 bytes (fp16)
  u32x4 wreg[kInt4 ? 1 : 4];
  half_t sreg = (half_t)0.0f;
  auto load_w = [&](int g) {
    if constexpr (kInt4) {
      wreg[0] = *(const u32x4*)(p.w + (int64_t)nc * p.w_stride + g * (kGroup / 2) + grp * 16);
      sreg = p.scales[(int64_t)nc * p.s_stride + g];
    } else {
      const half_t* wr = (const half_t*)p.w + (int64_t)nc * p.w_stride + g * kGroup + grp * 32;
#pragma unroll
      for (int s = 0; s < 4; ++s) wreg[s] = *(const u32x4*)(wr + 8 * s);
    }
  };

  floatx4 acc[kMSub];
#pragma unroll
  for (int j = 0; j < kMSub; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};

  if (g_begin < g_end) {
    load_x(g_begin);
    load_w(g_begin);
  }
  int buf = 0;
  for (int g = g_begin; g < g_end; ++g) {
    store_x(buf);
    __syncthreads();
    half8 wf[4];
    if constexpr (kInt4) {
      const half2_t s2 = {sreg, sreg};
#pragma unroll
      for (int s = 0; s < 4; ++s) wf[s] = dequant8(wreg[0][s], s2);
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) wf[s] = as_half8(wreg[s]);
    }
    if (g + 1 < g_end) {  // next group's loads overlap this group's MFMAs
      load_x(g + 1);
      load_w(g + 1);
    }
    const half_t* xb = &xs[buf][row * kLdsRow + grp * 32];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int j = 0; j < kMSub; ++j) {
        const half8 xf = as_half8(*(const u32x4*)(xb + j * 16 * kLdsRow + 8 * s));
        acc[j] = mfma16x16x32(wf[s], xf, acc[j]);
      }
    }
    buf ^= 1;
  }

  store_tile<kMSub>(p, acc, m0, blockIdx.x * kNTile);
}

// fp16 store of C[m][nb .. nb + 3] (columns past N dropped)
__device__ __forceinline__ void store_half4(const Params& p, floatx4 v, int m, int nb) {
  half_t* dst = p.out + (int64_t)m * p.out_stride + nb;
  const half4 h = to_half4(v);
  if (nb + 3 < p.N && ((uintptr_t)dst & 7) == 0) {
    *(half4*)dst = h;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (nb + i < p.N) dst[i] = h[i];
  }
}

// dequant8 with each mask-and-insert as one v_and_or_b32 (the mask from a scalar register,
// the fp16 exponent bits from a vector register): 18 VALU instructions per eight weights,
// the same values bit for bit.
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t bits) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
  return r;
}

__device__ __forceinline__ half8 dequant8_ao(uint32_t d, half2_t s2, uint32_t mask, uint32_t bits) {
#pragma clang fp contract(off)
  d ^= 0x88888888u;
  const uint32_t e = d >> 4;
  const uint32_t lo = __builtin_amdgcn_perm(e, d, 0x05040100u);
  const uint32_t hi = __builtin_amdgcn_perm(e, d, 0x07060302u);
  const half2_t bias = {(half_t)1032.0f, (half_t)1032.0f};
  u32x4 r;
  r[0] = as_u32((as_h2(and_or(lo, mask, bits)) - bias) * s2);
  r[1] = as_u32((as_h2(and_or(lo >> 8, mask, bits)) - bias) * s2);
  r[2] = as_u32((as_h2(and_or(hi, mask, bits)) - bias) * s2);
  r[3] = as_u32((as_h2(and_or(hi >> 8, mask, bits)) - bias) * s2);
  return as_half8(r);
}

// K split of a tile whose block b of wave w is acc[b] of every lane.  The workgroups of one tile
// have block ids congruent modulo 8, which the dispatcher places on one XCD (checked once per
// device before counters are handed out), so the tile's partial sums and its arrival counter
// are shared through that XCD's L2.  Each workgroup stores its partials
// ([tile][split][wave][block][lane]), waits until the stores are done and increments the tile's
// counter; the one that arrives last loads the other partials (bypassing L1), adds all of them
// in split order from 0 (the same sum whichever is last) and sets the counter back to zero for
// the next call.  No workgroup waits for another.  True for the last one, whose acc holds the
// sums.  `ti`: index of tile t among those of XCD group xg.
template <int kB>
__device__ __forceinline__ bool add_splits(const Params& p, floatx4 (&acc)[kB], int t, int s,
                                           int xg, int ti, int wave, int lane) {
  __shared__ unsigned arrived;
  floatx4* part = (floatx4*)p.partial + (int64_t)t * p.ksplit * (4 * kB * 64);
  floatx4* mine = part + ((int64_t)s * 4 + wave) * (kB * 64) + lane;
#pragma unroll
  for (int b = 0; b < kB; ++b) mine[b * 64] = acc[b];
  if (!p.counters) return false;  // no counters: a second launch adds the splits
  wait_vmcnt<0>();  // the stores are in L2 before the counter moves
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned* ctr = p.counters + xg * p.counter_stride + ti;
    const unsigned old = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (old == (unsigned)p.ksplit - 1)  // every other split has arrived: clear for the next call
      __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    arrived = old;
  }
  __syncthreads();
  if (arrived != (unsigned)p.ksplit - 1) return false;
  // the other splits' partials, loaded with sc0 (L1 bypassed), four blocks x four splits in
  // flight; own sums in place of split s
  const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
      part, (short)0, p.ksplit * 4 * kB * 1024, 0x00020000);
  constexpr int kBatch = kB < 4 ? kB : 4;
#pragma unroll
  for (int b0 = 0; b0 < kB; b0 += kBatch) {
    floatx4 sum[kBatch] = {};
    for (int s0 = 0; s0 < p.ksplit; s0 += 4) {
      floatx4 pv[kBatch][4] = {};
#pragma unroll
      for (int b = 0; b < kBatch; ++b)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (s0 + k < p.ksplit && s0 + k != s)
            pv[b][k] = __builtin_bit_cast(
                floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                             pr, ((((s0 + k) * 4 + wave) * kB + b0 + b) * 64 + lane) * 16, 0, 1));
#pragma unroll
      for (int b = 0; b < kBatch; ++b)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (s0 + k < p.ksplit) sum[b] += s0 + k == s ? acc[b0 + b] : pv[b][k];
    }
#pragma unroll
    for (int b = 0; b < kBatch; ++b) acc[b0 + b] = sum[b];
  }
  return true;
}

// The same sum for element `idx` of the partials (one thread each): tile t, place `at` in it.
template <int kB>
__device__ __forceinline__ floatx4 split_sum(const Params& p, int64_t idx, int& t, int& at) {
  at = (int)(idx % (4 * kB * 64));
  t = (int)(idx / (4 * kB * 64));
  const floatx4* part = (const floatx4*)p.partial + (int64_t)t * p.ksplit * (4 * kB * 64) + at;
  floatx4 sum = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < p.ksplit; ++s) sum += part[(int64_t)s * (4 * kB * 64)];
  return sum;
}

// ---------------------------------------------------------------------------------------
// Packed weights, unpacked inside the GEMM: from a few rows up to where one unpacking of the
// whole weight into memory costs less than unpacking it once per row tile (plan()).
//
// One workgroup of four waves per TM-row x 64 NB-column tile of C and K split; wave w owns all
// TM rows of columns 16 NB w .. 16 NB w + 16 NB - 1, so every weight is read and unpacked by one
// wave only, straight in registers, and an X fragment read from LDS feeds NB MFMAs.  Per
// 128-wide K group the tile's X rows are copied global -> LDS (buffer_load ... lds) into one of
// two stages while the other is multiplied; the next group's weights travel in registers at
// the same time.  LDS and registers leave room for two workgroups per CU (four of the smaller
// tiles), so one workgroup's wait at the group boundary is covered by another's MFMAs.
//
// X stage layout: two panels of 128 bytes per row (64 k each), 16-byte chunk c of row r at slot
// c ^ ((r / 2) % 8), so that the 16 rows a quarter-wave reads fall on distinct banks.  Lane
// group g supplies k = 32 g + 8 q .. +7 in k-step q: its 16 weight bytes of the group.
//
// Block ids congruent modulo 8 share an XCD: XCD e takes the e-th eighth of the column-major
// tile list, so a weight column tile is read by one XCD, and a tile's K splits meet in its L2
// (add_splits).
//
// What bounds it: at small M the weight stream and one memory latency per group; at large M
// the unpack (18 VALU instructions per eight weights beside TM / 16 MFMAs), which overlaps the
// MFMAs only in part.  3072 columns, K 8192, batches of layers with cold weights: 509 rows
// 157 -> 44 us against one unpacking pass and 256 x 256 tiles (24 of them for 256 CUs), 128
// rows 25.4 -> 17.8 us and 64 rows 18.8 -> 13.5 us against the kernels it replaces there.
template <int TM, int NB>
struct MidTile {
  static constexpr int kN = 64 * NB;           // columns per workgroup
  static constexpr int kMSub = TM / 16;
  static constexpr int kBlocks = NB * kMSub;   // 16 x 16 output blocks per wave
  static constexpr int kStage = TM * 256;      // LDS bytes of one group's X rows
};

template <int TM, int NB>
__global__ __launch_bounds__(kThreads, 2) void mid_gemm_kernel(Params p) {
  using T = MidTile<TM, NB>;
  constexpr int kMSub = T::kMSub;
  __shared__ __attribute__((aligned(16))) char lds[2 * T::kStage];

  const int t8 = (p.tiles + 7) >> 3;
  const int xg = blockIdx.x & 7, kk = blockIdx.x >> 3;
  const int s = __builtin_amdgcn_readfirstlane(kk / t8), ti = kk - s * t8;
  const int t_first = (int)((int64_t)xg * p.tiles >> 3);
  const int t = t_first + ti;
  if (t >= (int)((int64_t)(xg + 1) * p.tiles >> 3)) return;  // uniform, before any barrier
  const int tn = __builtin_amdgcn_readfirstlane(t / p.tiles_m), tm = t - tn * p.tiles_m;
  const int m0 = tm * TM;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15;
  const int grp = lane >> 4;
  const int nw = tn * T::kN + wave * 16 * NB;  // first column of this wave
  const int groups = p.K / kGroup;
  const int g_begin = s * p.groups_per_split;
  const int g_end = min(g_begin + p.groups_per_split, groups);

  // X rows past M read zeros through the buffer bounds
  const int rows_x = min(TM, p.M - m0);
  const rsrc_t xr = raw_rsrc(p.x + (int64_t)m0 * p.x_stride,
                             (int)(((int64_t)(rows_x - 1) * p.x_stride + p.K) * 2));
  // wave l fills its half (l / 2) of the rows of panel l % 2: copy i covers rows 8 i .. 8 i + 7
  // of them, lane l row l / 8, slot l % 8 <- chunk (l % 8) ^ ((r / 2) % 8)
  const int xr0 = (wave >> 1) * (TM / 2) + (lane >> 3);
  const int xrow = xr0 * (int)p.x_stride * 2 + (wave & 1) * 128;
  const int xoff0 = xrow + (((lane & 7) ^ ((xr0 >> 1) & 7)) << 4);
  const int xoff1 = xrow + (((lane & 7) ^ (((xr0 >> 1) + 4) & 7)) << 4);
  const int xstep = 8 * (int)p.x_stride * 2;
  const uint32_t lds0 = lds_addr(lds) + (wave & 1) * (TM * 128) + (wave >> 1) * (TM * 64);
  auto issue_x = [&](int buf, int g) {
    const int soff = __builtin_amdgcn_readfirstlane(g * 256);
#pragma unroll
    for (int i = 0; i < kMSub; ++i)
      lds_copy16(xr, lds0 + buf * T::kStage + i * 1024, ((i & 1) ? xoff1 : xoff0) + i * xstep, soff);
  };

  // this lane's weight rows (columns past N compute on the last row, never stored)
  struct Weights {
    u32x4 v[NB];
    uint32_t s[NB];  // scale bits
  };
  const uint8_t* wp[NB];
  const uint16_t* sp[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int64_t n = min(nw + 16 * j + row, p.N - 1);
    wp[j] = p.w + n * p.w_stride + grp * 16;
    sp[j] = (const uint16_t*)p.scales + n * p.s_stride;
  }
  auto load_w = [&](Weights& w, int g) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      w.v[j] = *(const u32x4*)(wp[j] + (int64_t)g * (kGroup / 2));
      w.s[j] = sp[j][g];
    }
  };

  floatx4 acc[T::kBlocks];  // block j * kMSub + i: columns 16 j.., rows 16 i.. of the wave's
#pragma unroll
  for (int b = 0; b < T::kBlocks; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};

  const uint32_t mask = __builtin_amdgcn_readfirstlane(0x000F000Fu);
  const uint32_t bits = 0x64006400u;
  // One group's MFMAs, software pipelined: the next k-step's X fragments are read and its
  // weights unpacked between this one's MFMAs (sched_group_barrier).
  auto compute = [&](int buf, const Weights& w) {
    half8 wf[2][NB], xf[2][kMSub];
    auto unpack = [&](int q) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
        wf[q & 1][j] = dequant8_ao(w.v[j][q], as_h2(w.s[j] * 0x10001u), mask, bits);
    };
    auto read = [&](int q) {
      const int ch = 4 * grp + q;
      const char* pa = lds + buf * T::kStage + (ch >> 3) * (TM * 128) + row * 128 +
                       (((ch & 7) ^ ((row >> 1) & 7)) << 4);
#pragma unroll
      for (int i = 0; i < kMSub; ++i) xf[q & 1][i] = as_half8(*(const u32x4*)(pa + i * 2048));
    };
    read(0);
    unpack(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < 3) {
        read(q + 1);
        unpack(q + 1);
      }
#pragma unroll
      for (int i = 0; i < kMSub; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[j * kMSub + i] = mfma16x16x32(wf[q & 1][j], xf[q & 1][i], acc[j * kMSub + i]);
      if (q < 3) {
#pragma unroll
        for (int i = 0; i < kMSub; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one fragment read
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, (20 + kMSub - 1) / kMSub, 0);  // VALU
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // every wave has landed its part of this group's X and its weights, and is done reading
  // the other stage
  auto boundary = [&] {
    wait_vmcnt<0>();
    wait_lgkmcnt0();
    asm volatile("s_barrier" ::: "memory");
  };

  Weights wa, wb;
  load_w(wa, g_begin);
  issue_x(0, g_begin);
  for (int g = g_begin; g < g_end; g += 2) {
    boundary();
    if (g + 1 < g_end) {
      load_w(wb, g + 1);
      issue_x(1, g + 1);
    }
    compute(0, wa);
    if (g + 1 >= g_end) break;
    boundary();
    if (g + 2 < g_end) {
      load_w(wa, g + 2);
      issue_x(0, g + 2);
    }
    compute(1, wb);
  }

  if (p.ksplit > 1 && !add_splits<T::kBlocks>(p, acc, t, s, xg, ti, wave, lane)) return;
#pragma unroll
  for (int i = 0; i < kMSub; ++i) {
    const int m = m0 + 16 * i + row;
    if (m < p.M) {
#pragma unroll
      for (int j = 0; j < NB; ++j) store_half4(p, acc[j * kMSub + i], m, nw + 16 * j + 4 * grp);
    }
  }
}

// mid_gemm_kernel's split sums in a second launch, for streams without arrival counters: the
// same additions in the same order.  One thread per (tile, wave, block, lane).
template <int TM, int NB>
__global__ __launch_bounds__(256) void mid_reduce_kernel(Params p) {
  using T = MidTile<TM, NB>;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p.tiles * 4 * T::kBlocks * 64) return;
  int t, at;
  const floatx4 sum = split_sum<T::kBlocks>(p, idx, t, at);
  const int lane = at & 63, b = (at >> 6) % T::kBlocks, wave = at / (64 * T::kBlocks);
  const int tn = t / p.tiles_m, tm = t - tn * p.tiles_m;
  const int m = tm * TM + 16 * (b % T::kMSub) + (lane & 15);
  if (m < p.M)
    store_half4(p, sum, m, tn * T::kN + wave * 16 * NB + 16 * (b / T::kMSub) + 4 * (lane >> 4));
}

// ---------------------------------------------------------------------------------------
// fp16 weights from 5 rows, and packed weights unpacked once into the workspace where the row
// tiles are many (mid_gemm_kernel spends a third of its time unpacking there).
//
// C[M, N] = X[M, K] * W[N, K]^T, fp16 in and out, fp32 accumulation, K a multiple of 128.
// One workgroup per 32 BM x 32 BN tile of C (and K split), four waves, one per SIMD.  Wave w
// owns 16 BM rows (m, 16 BM * (w / 2)..) x 16 BN columns (n, 16 BN * (w % 2)..) of the tile: BM x
// BN MFMA tiles of v_mfma_f32_16x16x32_f16, W as the A operand and X^T as the B operand.  Per
// 64-wide K step the tile's X and W rows (128 bytes each, 16-byte chunk c of row r at slot
// c ^ ((r / 2) % 8), so the 16 rows a quarter-wave reads fall on distinct banks) are copied
// global -> LDS with buffer_load ... lds into one of S stages, S - 1 steps ahead.  A step is two
// k-substeps: the second substep's fragments are read between the first substep's MFMAs; after
// three quarters of the second substep's MFMAs the wave waits for its copies of the next step
// and passes a barrier (every wave has then read this step's stage and landed the next), and
// the next step's first fragments are read between the last quarter.  The copies go out between
// the first substep's MFMAs, into the stage every wave finished reading before the previous
// step's barrier.
//
// Tiles: 256 x 256 (256 fp32 sums per lane in the AGPRs, each fragment feeds eight MFMAs, one
// workgroup per CU) reaches the highest rate, 1.35 PFLOP/s when its tiles fill whole rounds of
// the CUs; the smaller ones, two workgroups per CU with two to five stages, fill the chip when
// those tiles are too few (3072 columns, K 8192: 509 rows 160 -> 43 us with 128 x 128 tiles and
// four K splits; 100 rows x 3072 columns, K 3072: 30 -> 11 us with 64 x 64 and four).
constexpr int kGemmK = 64;              // K per step
constexpr int kGemmRowB = kGemmK * 2;   // bytes per LDS row

// Tile of the fp16 GEMM: four waves, two by two, each 16 BM rows x 16 BN columns; S LDS stages.
template <int BM, int BN, int S>
struct GemmTile {
  static constexpr int kM = 32 * BM, kN = 32 * BN;      // rows and columns of C per workgroup
  static constexpr int kXB = kM * kGemmRowB;            // X rows of one step
  static constexpr int kStage = kXB + kN * kGemmRowB;   // X rows, then W rows
  static constexpr int kBlocks = BM * BN;               // 16 x 16 output blocks per wave
  static constexpr int kOps = BM + BN;                  // copies (and fragments) per wave
  static constexpr bool kSplit = kBlocks < 64;          // K splits (256 x 256 tiles take none)
  static constexpr int kPerCu = S * kStage <= 80 * 1024 ? 2 : 1;  // workgroups per CU
  static_assert(4 * 16 * BM * 32 * BN <= S * kStage, "the staged output fits the stages");
};

template <int BM, int BN, int S>
__global__ __launch_bounds__(kThreads, (GemmTile<BM, BN, S>::kPerCu)) void tile_gemm_kernel(Params p) {
  using T = GemmTile<BM, BN, S>;
  __shared__ __attribute__((aligned(16))) char lds[S * T::kStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1;  // wave tile: columns 16 BN wn.., rows 16 BM wm..
  // Tile order: block id L runs on XCD L % 8.  With p.band XCD e takes row tiles e * band ..
  // e * band + band - 1 against every column tile (the X rows of its tiles stay in its own
  // L2); otherwise 256 x 256 tiles in column-major order over all XCDs, which read a column's W
  // rows at the same time (16000 x 2048, K 8192 505 -> 436 us against the order below), and
  // smaller ones XCD e the e-th eighth of that list (its W rows stay in its L2, and a tile's K
  // splits meet there).
  const int xg = blockIdx.x & 7, kk = blockIdx.x >> 3;
  int tm, tn, s = 0, ti = 0, t = 0;
  if (p.band) {
    tm = xg * p.band + kk % p.band;
    tn = kk / p.band;
  } else {
    if constexpr (T::kSplit) {
      const int t8 = (p.tiles + 7) >> 3;
      s = __builtin_amdgcn_readfirstlane(kk / t8);
      ti = kk - s * t8;
      t = (int)((int64_t)xg * p.tiles >> 3) + ti;
      if (t >= (int)((int64_t)(xg + 1) * p.tiles >> 3)) return;  // uniform, before any barrier
    } else {
      t = blockIdx.x;
      if (t >= p.tiles) return;
    }
    tn = t / p.tiles_m;
    tm = t - tn * p.tiles_m;
  }
  tm = __builtin_amdgcn_readfirstlane(tm);
  tn = __builtin_amdgcn_readfirstlane(tn);
  const int m0 = tm * T::kM, n0 = tn * T::kN;
  const int rows_x = min(T::kM, p.M - m0), rows_w = min(T::kN, p.N - n0);
  // descriptors over exactly the tile's rows: lanes of rows past M or N read zeros
  const rsrc_t xr = raw_rsrc(p.x + (int64_t)m0 * p.x_stride,
                             (int)(((int64_t)(rows_x - 1) * p.x_stride + p.K) * 2));
  const rsrc_t wr = raw_rsrc((const half_t*)p.w + (int64_t)n0 * p.w_stride,
                             (int)(((int64_t)(rows_w - 1) * p.w_stride + p.K) * 2));
  // this wave copies a quarter of the X rows and of the W rows, eight rows an instruction;
  // lane l fills slot l % 8 of row r0 + l / 8 with chunk (l % 8) ^ ((r / 2) % 8)
  int xoff[BM], woff[BN];
#pragma unroll
  for (int i = 0; i < BM; ++i) {
    const int r = 8 * (BM * wave + i) + (lane >> 3);
    xoff[i] = r < rows_x ? (int)((int64_t)r * p.x_stride * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4)
                         : 0x7ffffff0;
  }
#pragma unroll
  for (int i = 0; i < BN; ++i) {
    const int r = 8 * (BN * wave + i) + (lane >> 3);
    woff[i] = r < rows_w ? (int)((int64_t)r * p.w_stride * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4)
                         : 0x7ffffff0;
  }
  const uint32_t lds0 = lds_addr(lds);
  const int k0 = 2 * s * p.groups_per_split;  // first step (two per 128-wide group)
  const int steps = min(2 * p.groups_per_split, p.K / kGemmK - k0);
  // copy q of step kt into stage st: X rows for q < BM, W rows for q >= BM
  auto copy = [&](int kt, int st, int q) {
    const uint32_t base = lds0 + st * T::kStage;
    const int soff = __builtin_amdgcn_readfirstlane((k0 + kt) * kGemmRowB);
    if (q < BM)
      lds_copy16(xr, base + 8 * (BM * wave + q) * kGemmRowB, xoff[q < BM ? q : 0], soff);
    else
      lds_copy16(wr, base + T::kXB + 8 * (BN * wave + q - BM) * kGemmRowB,
                 woff[q < BM ? 0 : q - BM], soff);
  };

  floatx4 acc[T::kBlocks];  // block i * BM + j: columns 16 i.., rows 16 j.. of the wave's tile
#pragma unroll
  for (int b = 0; b < T::kBlocks; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};

  // fragment q of k-substep h: W tile q (q < BN) or X tile q - BN, row 16 * tile + fr, chunk
  // 4h + fg; rows 16i + fr share (row / 2) % 8 with row fr
  const int fr = lane & 15, fg = lane >> 4;
  const int sw = (fr >> 1) & 7;
  const int xrow0 = (16 * BM * wm + fr) * kGemmRowB;
  const int wrow0 = T::kXB + (16 * BN * wn + fr) * kGemmRowB;
  auto frag = [&](const char* st, int h, int q) {
    const int row0 = q < BN ? wrow0 + q * 16 * kGemmRowB : xrow0 + (q - BN) * 16 * kGemmRowB;
    return as_half8(*(const u32x4*)(st + row0 + (((4 * h + fg) ^ sw) << 4)));
  };
  half8 f0[T::kOps], f1[T::kOps];
  // the scheduler keeps each group of MFMAs with its reads and copies (sched_barrier)
  auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
  auto mfmas = [&](half8 (&f)[T::kOps], int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1; ++e) acc[e] = mfma16x16x32(f[e / BM], f[BN + e % BM], acc[e]);
  };

#pragma unroll
  for (int d = 0; d < S - 1; ++d)
    if (d < steps) {
#pragma unroll
      for (int q = 0; q < T::kOps; ++q) copy(d, d, q);
    }
  if (steps >= S - 1)
    wait_vmcnt<(S - 2) * T::kOps>();
  else
    wait_vmcnt<0>();
  asm volatile("s_barrier" ::: "memory");
  fence();
#pragma unroll
  for (int q = 0; q < T::kOps; ++q) f0[q] = frag(lds, 0, q);
  fence();
  int cur = 0, fill = S - 1;  // stages of this step and of the step the copies go to
  // kMore: a step follows; kFill: step kt + S - 1 exists
  auto step = [&](int kt, auto more_c, auto fill_c) {
    constexpr bool kMore = decltype(more_c)::value, kFill = decltype(fill_c)::value;
    const char* st = lds + cur * T::kStage;
    // substep 0 on f0; substep 1's fragments read and step kt + S - 1's copies issued
#pragma unroll
    for (int g = 0; g < T::kOps; ++g) {
      f1[g] = frag(st, 1, g);
      if constexpr (kFill) copy(kt + S - 1, fill, g);
      mfmas(f0, g * T::kBlocks / T::kOps, (g + 1) * T::kBlocks / T::kOps);
      fence();
    }
    // substep 1 on f1: three quarters of its MFMAs, the wait and barrier, then the last
    // quarter with the next step's substep-0 fragments read between them
    constexpr int kQ = T::kBlocks * 3 / 4;
#pragma unroll
    for (int e = 0; e < kQ; e += 4) {
      mfmas(f1, e, e + 4 < kQ ? e + 4 : kQ);
      fence();
    }
    if constexpr (kMore) {
      wait_vmcnt<kFill ? (S - 2) * T::kOps : 0>();
      wait_lgkmcnt0();
      asm volatile("s_barrier" ::: "memory");
      fence();
    }
    cur = cur + 1 == S ? 0 : cur + 1;
    fill = fill + 1 == S ? 0 : fill + 1;
    const char* nst = lds + cur * T::kStage;
    constexpr int kR = T::kBlocks - kQ < 4 ? T::kBlocks - kQ : 4;  // read groups
#pragma unroll
    for (int g = 0; g < kR; ++g) {
      if constexpr (kMore) {
#pragma unroll
        for (int u = g * T::kOps / kR; u < (g + 1) * T::kOps / kR; ++u) f0[u] = frag(nst, 0, u);
      }
      mfmas(f1, kQ + g * (T::kBlocks - kQ) / kR, kQ + (g + 1) * (T::kBlocks - kQ) / kR);
      fence();
    }
  };
  int kt = 0;
  for (; kt + S - 1 < steps; ++kt) step(kt, std::true_type{}, std::true_type{});
  for (; kt + 1 < steps; ++kt) step(kt, std::true_type{}, std::false_type{});
  step(steps - 1, std::false_type{}, std::false_type{});

  if constexpr (T::kSplit)
    if (p.ksplit > 1 && !add_splits<T::kBlocks>(p, acc, t, s, xg, ti, wave, lane)) return;
  wait_lgkmcnt0();
  __syncthreads();  // every wave is done with the stages
  fence();

  // Lane (m = 16j + fr, fg) holds C[m][16i + 4fg .. +3] of the wave's tile.  Rows go through
  // the wave's own part of the LDS (fp16, chunk c of row m at c ^ (m % chunks)) so that whole
  // rows of the wave's tile are stored by consecutive lanes.
  constexpr int kRow = 32 * BN, kCh = 2 * BN;
  char* cs = lds + wave * (16 * BM * kRow);
#pragma unroll
  for (int j = 0; j < BM; ++j) {
    const int m = 16 * j + fr;
#pragma unroll
    for (int i = 0; i < BN; ++i) {
      const int c = 2 * i + (fg >> 1);
      *(half4*)(cs + m * kRow + ((c ^ (m & (kCh - 1))) << 4) + ((fg & 1) << 3)) =
          to_half4(acc[i * BM + j]);
    }
  }
  wave_lds_sync();
  const int sr = lane / kCh, sc = lane % kCh;
  const int gn = n0 + 16 * BN * wn + 8 * sc;
#pragma unroll 4
  for (int q = 0; q < 16 * BM * kCh / 64; ++q) {
    const int m = (64 / kCh) * q + sr;
    const u32x4 v = *(const u32x4*)(cs + m * kRow + ((sc ^ (m & (kCh - 1))) << 4));
    const int gm = m0 + 16 * BM * wm + m;
    if (gm >= p.M || gn >= p.N) continue;
    half_t* dst = p.out + (int64_t)gm * p.out_stride + gn;
    if (p.vec_out) {
      *(u32x4*)dst = v;
    } else {
      const half8 h = as_half8(v);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (gn + e < p.N) dst[e] = h[e];
    }
  }
}

// tile_gemm_kernel's split sums in a second launch, for streams without arrival counters: the
// same additions in the same order.  One thread per (tile, wave, block, lane).
template <int BM, int BN>
__global__ __launch_bounds__(256) void tile_reduce_kernel(Params p) {
  constexpr int kB = BM * BN;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p.tiles * 4 * kB * 64) return;
  int t, at;
  const floatx4 sum = split_sum<kB>(p, idx, t, at);
  const int lane = at & 63, b = (at >> 6) % kB, wave = at / (64 * kB);
  const int tn = t / p.tiles_m, tm = t - tn * p.tiles_m;
  const int m = tm * 32 * BM + (wave >> 1) * 16 * BM + 16 * (b % BM) + (lane & 15);
  if (m < p.M)
    store_half4(p, sum, m, tn * 32 * BN + (wave & 1) * 16 * BN + 16 * (b / BM) + 4 * (lane >> 4));
}

// A barrier for data passed through LDS only: __syncthreads would also wait for the weight loads
// in flight.
__device__ __forceinline__ void lds_barrier() {
  wait_lgkmcnt0();
  asm volatile("s_barrier" ::: "memory");
}

// Decode-sized calls (16 rows of X per blockIdx.y): one workgroup per 16 output columns.
// The kW waves take interleaved groups (g = wave, wave + kW, ...), so K is split inside
// the workgroup and no partials leave it.  Each lane issues the loads of kChunk groups at
// once (16 weight bytes, the scale, and 64 bytes of its X row per group) before any math,
// so one memory latency covers the chunk; the kW waves' sums are added through LDS in
// a fixed order.
//
// kNormRows > 0: the RMSNorm of up to that many rows fused, shared out over the workgroup (packed
// weights, 1 row, or 2 of more than kShortRow elements) or a row per wave.  5120 columns, K 3072,
// packed, cold weights: 1 row 8.0 us, 8.8 a row per wave; 16384 columns 12.2 against 15.2 and, 2
// rows, 13.6 against 15.1.  4 rows shared out take 10.9 against 9.1, 2 short rows leave most
// threads idle (7168 columns, K 256 6.2 against 5.6), and fp16 weights, bound by their stream,
// lose too.
constexpr int kShortRow = 1024;
template <bool kInt4, int kChunk, int kNormRows, int kW>
__global__ __launch_bounds__(64 * kW, kNormRows == kFusedNormM ? 1 : 2) void gemv_kernel(Params p) {
  constexpr bool kNorm = kNormRows > 0;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row = lane & 15;
  const int grp = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int n = n0 + row;
  const int nc = n < p.N ? n : p.N - 1;
  const int m = blockIdx.y * 16 + row;  // the X row this lane supplies
  const bool m_ok = m < p.M;
  // MFMA output column j depends on X row j only, and the columns of rows past M are never
  // stored: those lanes read zeros (or, from the normalized rows in LDS, a valid row)
  const int groups = p.K / kGroup;
  // fused norm: the workgroup's (at most 16, in practice a few) rows are normalized once
  // into LDS, [rows, K] fp16, and the X operand is read from there
  extern __shared__ __attribute__((aligned(16))) half_t xn[];
  const int rows_n = min(16, p.M - (int)blockIdx.y * 16);
  const half_t* xrow_n = xn + min(row, rows_n - 1) * p.K;

  // Issue the loads of one chunk (kChunk groups of this wave, g0, g0 + kW, ...): every load
  // goes out before any math and without branches (groups past the end reload the last
  // group and are skipped), so one latency covers the chunk.
  u32x4 wv[kInt4 ? kChunk : 4 * kChunk];
  half_t sv[kChunk];
  u32x4 xv[kNorm ? 1 : 4 * kChunk];
  // X through a buffer descriptor over this workgroup's rows: lanes of rows past M use an
  // offset past the end and read zeros with no memory request and no branch (the host
  // rejects calls whose 16 rows span more than 0x7ffffff0 bytes)
  const __amdgpu_buffer_rsrc_t xr_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.x + (int64_t)blockIdx.y * 16 * p.x_stride), (short)0,
      (int)(((int64_t)(rows_n - 1) * p.x_stride + p.K) * 2), 0x00020000);
  const int x_off0 = m_ok ? (int)(((int64_t)row * p.x_stride + grp * 32) * 2) : 0x7ffffff0;
  auto load_chunk = [&](int g0) {
#pragma unroll
    for (int c = 0; c < kChunk; ++c) {
      const int g = min(g0 + kW * c, groups - 1);
      if constexpr (kInt4) {
        wv[c] = *(const u32x4*)(p.w + (int64_t)nc * p.w_stride + g * (kGroup / 2) + grp * 16);
        sv[c] = p.scales[(int64_t)nc * p.s_stride + g];
      } else {
        const half_t* wr = (const half_t*)p.w + (int64_t)nc * p.w_stride + g * kGroup + grp * 32;
#pragma unroll
        for (int s = 0; s < 4; ++s) wv[4 * c + s] = *(const u32x4*)(wr + 8 * s);
      }
      if constexpr (!kNorm) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          xv[4 * c + s] = __builtin_bit_cast(
              u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                         xr_rsrc, m_ok ? x_off0 + (g * kGroup + 8 * s) * 2 : x_off0, 0, 0));
      }
    }
  };

  // the first chunk's weights are in flight while the rows are normalized; the scheduling
  // barriers keep every load of a chunk ahead of its math (the scheduler would otherwise
  // start the math after the first few loads and issue the rest one latency later)
  if constexpr (kNorm && kNormRows < kFusedNormM) {
    // Every thread takes a few elements of every row: a row's sum of squares is the sum of the
    // waves' parts (through LDS), and no wave holds a whole row in registers, so two
    // eight-wave workgroups fit a CU.  x and the norm weight are loaded before the first
    // chunk's weights: loads complete in issue order, so the norm waits for its own data only
    // and runs while the weights stream in.  Rows longer than kLongRow are normalized after
    // the weights' loads, a wave per row.
    constexpr int kLongRow = 8192, kSpan = kW * 512, kParts = kLongRow / kSpan;
    if (p.K <= kLongRow) {  // uniform
      __shared__ float part[kNormRows][kW];
      u32x4 xr_v[kNormRows][kParts], nw_v[kParts];
      // elements past K and rows past M read zeros through the buffer bounds
      const __amdgpu_buffer_rsrc_t nw_rsrc =
          __builtin_amdgcn_make_buffer_rsrc((void*)p.norm_w, (short)0, p.K * 2, 0x00020000);
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        const int k2 = (threadIdx.x * 8 + i * kSpan) * 2;
#pragma unroll
        for (int r = 0; r < kNormRows; ++r)
          xr_v[r][i] = __builtin_bit_cast(
              u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                         xr_rsrc, k2 < 2 * p.K && r < rows_n ? r * (int)(p.x_stride * 2) + k2 : 0x7ffffff0,
                         0, 0));
        nw_v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(nw_rsrc, k2, 0, 0));
      }
      load_chunk(wave);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < kNormRows; ++r) {
        float sq = 0.f;
#pragma unroll
        for (int i = 0; i < kParts; ++i) sq += sum_sq8(xr_v[r][i]);
        sq = wave_sum(sq);
        if (lane == 0) part[r][wave] = sq;
      }
      lds_barrier();
#pragma unroll
      for (int r = 0; r < kNormRows; ++r) {
        if (r < rows_n) {  // uniform
          float sq = 0.f;
#pragma unroll
          for (int w = 0; w < kW; ++w) sq += part[r][w];
          const float rs = rsqrtf(sq / (float)p.K + p.eps);
#pragma unroll
          for (int i = 0; i < kParts; ++i) {
            const int k = threadIdx.x * 8 + i * kSpan;
            if (k < p.K) *(u32x4*)(xn + r * p.K + k) = norm8(xr_v[r][i], rs, nw_v[i]);
          }
        }
      }
    } else {
      load_chunk(wave);
      __builtin_amdgcn_sched_barrier(0);
      for (int r = wave; r < rows_n; r += kW)
        norm_row_to(p.x + (int64_t)(blockIdx.y * 16 + r) * p.x_stride, p.norm_w, p.K, p.eps,
                    xn + r * p.K, lane);
    }
    lds_barrier();
  } else if constexpr (kNorm) {
    // Wave r normalizes row r.  Its x row and the norm weight are loaded before the first
    // chunk's weights: loads complete in issue order, so the norm waits for its own data
    // only and runs while the weights stream in.  Rows longer than kRowChunks * 512, and rows
    // past the kW-th, are normalized after the weights' loads by norm_row_to.
    const bool in_regs = p.K <= kRowChunks * 512 && wave < rows_n;  // uniform
    u32x4 xr_v[kRowChunks], nw_v[kRowChunks];
    if (in_regs) {
      const half_t* xrow = p.x + (int64_t)(blockIdx.y * 16 + wave) * p.x_stride;
#pragma unroll
      for (int i = 0; i < kRowChunks; ++i) {
        const int k = lane * 8 + i * 512;
        xr_v[i] = k < p.K ? *(const u32x4*)(xrow + k) : u32x4{0, 0, 0, 0};
        nw_v[i] = k < p.K ? *(const u32x4*)(p.norm_w + k) : u32x4{0, 0, 0, 0};
      }
    }
    load_chunk(wave);
    __builtin_amdgcn_sched_barrier(0);
    if (in_regs) {
      float sq = 0.f;
#pragma unroll
      for (int i = 0; i < kRowChunks; ++i) sq += sum_sq8(xr_v[i]);
      const float r = rsqrtf(wave_sum(sq) / (float)p.K + p.eps);
#pragma unroll
      for (int i = 0; i < kRowChunks; ++i) {
        const int k = lane * 8 + i * 512;
        if (k < p.K) *(u32x4*)(xn + wave * p.K + k) = norm8(xr_v[i], r, nw_v[i]);
      }
    }
    for (int r = in_regs ? wave + kW : wave; r < rows_n; r += kW)
      norm_row_to(p.x + (int64_t)(blockIdx.y * 16 + r) * p.x_stride, p.norm_w, p.K, p.eps,
                  xn + r * p.K, lane);
    __syncthreads();
  } else {
    load_chunk(wave);
    __builtin_amdgcn_sched_barrier(0);
  }

  // two accumulators, alternating by k-step, halve the chain of dependent MFMAs
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  floatx4 acc2 = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int g0 = wave; g0 < groups; g0 += kW * kChunk) {
    if (g0 != wave) {
      load_chunk(g0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < kChunk; ++c) {
      if (g0 + kW * c < groups) {  // uniform across the wave
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          half8 wf;
          if constexpr (kInt4)
            wf = dequant8(wv[c][s], half2_t{sv[c], sv[c]});
          else
            wf = as_half8(wv[4 * c + s]);
          u32x4 xf;
          if constexpr (kNorm)
            xf = *(const u32x4*)(xrow_n + (g0 + kW * c) * kGroup + grp * 32 + 8 * s);
          else
            xf = xv[4 * c + s];
          if (s & 1)
            acc2 = mfma16x16x32(wf, as_half8(xf), acc2);
          else
            acc = mfma16x16x32(wf, as_half8(xf), acc);
        }
      }
      // one group's operands at a time: unbounded hoisting of the X reads and the
      // dequantization ahead of the MFMAs would spill
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  acc += acc2;

  __shared__ floatx4 red[kW][64];
  red[wave][lane] = acc;
  __syncthreads();
  if (wave == 0) {
    floatx4 t = red[0][lane];
#pragma unroll
    for (int w = 1; w < kW; ++w) t += red[w][lane];
    if (m_ok) {
      const int nb = n0 + 4 * grp;
      half_t* dst = p.out + (int64_t)m * p.out_stride + nb;
      const half4 h = to_half4(t);
      if (nb + 3 < p.N && ((uintptr_t)dst & 7) == 0) {
        *(half4*)dst = h;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < p.N) dst[i] = h[i];
      }
    }
  }
}

// out[m, n] = fp16(sum over splits of partial[s, m, n]), splits added in order.
__global__ __launch_bounds__(256) void reduce_kernel(const float* partial, int splits, int M,
                                                     int N, half_t* out, int64_t out_stride) {
  const int64_t total = (int64_t)M * N;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    float s = 0.f;
    for (int k = 0; k < splits; ++k) s += partial[k * total + i];
    const int64_t m = i / N;
    out[m * out_stride + (i - m * N)] = (half_t)s;
  }
}

// ---------------------------------------------------------------------------------------
// loader.py:9-41: symmetric groupwise INT4 quantization, with the reference's fp16 tensor
// arithmetic: amax = max|w| over the group (fp16), clamped below at fp16(1e-6); scale =
// fp16(fp32(amax) * fp32(1/7)) (torch multiplies by the reciprocal when a CUDA tensor is
// divided by a Python scalar); q = round_half_even(fp16(fp32(w) / fp32(scale))), clamped to
// [-8, 7].  gs / 8 lanes per group (gs a power of two from 8 to 512), 8 values per lane;
// a group's lanes are consecutive lanes of one wave, so they enter and leave the loop together.
__global__ __launch_bounds__(256) void quantize_kernel(const half_t* w, int64_t w_stride, int N,
                                                       int K, int gs, uint8_t* packed,
                                                       int64_t p_stride, half_t* scales,
                                                       int64_t s_stride) {
  const int groups = K / gs;
  const int lanes = gs / 8;          // per group
  const int shift = __builtin_ctz(lanes);
  const int64_t total = (int64_t)N * groups;
  const int lane16 = threadIdx.x & (lanes - 1);
  for (int64_t gi = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> shift; gi < total;
       gi += ((int64_t)gridDim.x * blockDim.x) >> shift) {
    const int nrow = (int)(gi / groups);
    const int g = (int)(gi - (int64_t)nrow * groups);
    const half8 v = as_half8(
        *(const u32x4*)(w + (int64_t)nrow * w_stride + (int64_t)g * gs + lane16 * 8));
    float amax = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf((float)v[e]));
    for (int d = 1; d < lanes; d <<= 1) amax = fmaxf(amax, __shfl_xor(amax, d, lanes));
    const float lo = (float)(half_t)1e-6f;
    amax = fmaxf(amax, lo);
    const half_t scale = (half_t)(amax * (1.0f / 7.0f));
    const float sf = (float)scale;
    uint32_t word = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float qf = (float)(half_t)((float)v[e] / sf);
      const float qr = fminf(fmaxf(__builtin_rintf(qf), -8.f), 7.f);
      word |= ((uint32_t)(int)qr & 0xFu) << (4 * e);
    }
    *(uint32_t*)(packed + (int64_t)nrow * p_stride + (int64_t)g * (gs / 2) + lane16 * 4) = word;
    if (lane16 == 0) scales[(int64_t)nrow * s_stride + g] = scale;
  }
}

// matmul.py:309-326 (_dequant_storage): W = fp16(q * scale), 8 values per thread (gs, the
// group size, a multiple of 8).
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t* packed, int64_t p_stride,
                                                         const half_t* scales, int64_t s_stride,
                                                         int N, int K, int gs, half_t* w,
                                                         int64_t w_stride) {
  const int per_row = K / 8;
  const int64_t total = (int64_t)N * per_row;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int nrow = (int)(i / per_row);
    const int c = (int)(i - (int64_t)nrow * per_row);
    const uint32_t d = *(const uint32_t*)(packed + (int64_t)nrow * p_stride + c * 4);
    const half_t s = scales[(int64_t)nrow * s_stride + (c * 8) / gs];
    *(u32x4*)(w + (int64_t)nrow * w_stride + c * 8) = as_u32x4(dequant8(d, half2_t{s, s}));
  }
}

// Kernel, tile and split count for an (M, N, K) call; shared by the size query and the launch.
struct Plan {
  bool gemv;    // gemv_kernel; otherwise mt x nt tiles:
  bool dense;   // tile_gemm_kernel (packed weights are first unpacked into the workspace), or
                // mid_gemm_kernel
  int mt, nt;
  int splits;
};

// Rows from which a call may use the dense 256 x 256 tiles; below, X rows may be any distance
// apart, from here 256 rows of X (and of an fp16 W) have to span less than 2 GiB.
constexpr int kDenseMinM = 129;
constexpr int kGemvMaxM = 16;    // rows of one gemv_kernel workgroup
constexpr int kMaxSplits = 16;
constexpr int kMaxSplitTiles = 8 * kXcdCounters;  // tiles of a split call
constexpr int64_t kMaxTiles = (1 << 24) - 8;      // of any: 2^32 threads a launch dimension

// Time of a call with one tile shape, in us, as measured on MI355X and fitted by least squares:
// 8232 sizes of 1 to 30000 rows, 88 to 28672 columns and K 128 to 14336, cold weights, each with
// every tile and several K splits.  The plan chosen by it is within 1% of the fastest on average,
// on sizes left out of the fit too, and within 6% for 19 of 20 (timings and fit:
// profiles/linear_plans.py).  Tables fitted to K 3072 and 8192 alone lost elsewhere (fp16 weights,
// K 384, 17 rows x 7168 columns 6.1 -> 10.5 us on 128 x 128 tiles; 5.2 with these):
//   fixed + per_wg x (workgroups on a CU - 1) + per_mb x weight MB + per_x_mb x MB of X read by
//   all column tiles + groups per split x (full rounds x load[per_cu] + load[workgroups of the
//   last round on a CU]) + (K split: split + per_split x splits)
// where a round is per_cu workgroups on every CU, and load[n] the time of one 128-wide K group
// with n workgroups on the CU.  A CU's workgroups are those of its XCD, which takes an eighth of
// the tiles.
struct TileCost {
  bool dense;
  int mt, nt, per_cu;
  float fixed, load[5], split, per_split, per_wg, per_mb, per_x_mb;
};
constexpr TileCost kPackedTiles[] = {
    {false, 16, 64, 4, 3.127f, {0, 0.303f, 0.363f, 0.452f, 0.574f}, 0.753f, 0.112f, 0.244f, 0.1381f, 0.0689f},
    {false, 32, 64, 4, 3.261f, {0, 0.354f, 0.418f, 0.577f, 0.764f}, 0.898f, 0.154f, 0.321f, 0.126f, 0.0444f},
    {false, 64, 64, 4, 3.567f, {0, 0.443f, 0.527f, 0.843f, 1.013f}, 1.34f, 0.256f, 0.521f, 0.0904f, 0.0384f},
    {false, 64, 128, 4, 4.225f, {0, 0.718f, 1.038f, 1.469f, 1.754f}, 1.788f, 0.539f, 1.078f, 0.0836f, 0.0528f},
    {false, 128, 64, 2, 4.099f, {0, 0.645f, 0.854f}, 2.06f, 0.547f, 1.366f, 0.0661f, 0.0344f},
    {false, 128, 128, 2, 5.345f, {0, 1.033f, 1.365f}, 3.251f, 0.971f, 2.677f, 0.0711f, 0.0484f},
    {true, 128, 128, 2, 5.226f, {0, 1.208f, 1.071f}, 0, 0, 1.92f, 0.0f, 0.0436f},
    {true, 256, 256, 1, 12.287f, {0, 1.788f}, 0, 0, 9.089f, 0.0164f, 0.0677f},
};
constexpr TileCost kHalfTiles[] = {
    {true, 32, 64, 2, 3.518f, {0, 0.24f, 0.428f}, 0.886f, 0.145f, 0.516f, 0.1152f, 0.0414f},
    {true, 64, 64, 2, 3.662f, {0, 0.288f, 0.459f}, 1.122f, 0.251f, 0.77f, 0.1064f, 0.0509f},
    {true, 64, 128, 2, 3.795f, {0, 0.482f, 0.763f}, 1.778f, 0.56f, 0.988f, 0.1196f, 0.0739f},
    {true, 128, 64, 2, 3.85f, {0, 0.486f, 0.706f}, 1.952f, 0.571f, 1.141f, 0.104f, 0.0406f},
    {true, 128, 128, 2, 4.227f, {0, 1.206f, 1.044f}, 3.66f, 1.0f, 2.255f, 0.0987f, 0.0698f},
    {true, 256, 256, 1, 11.089f, {0, 1.926f}, 0, 0, 9.416f, 0.1499f, 0.0699f},
};

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

inline float weight_mb(int64_t N, int64_t K, bool packed) { return (packed ? 0.5e-6f : 2e-6f) * N * K; }

inline float tile_cost(const TileCost& t, int64_t M, int64_t N, int64_t K, int64_t splits, bool int4,
                       int cus) {
  const int64_t tiles_n = ceil_div(N, t.nt), tiles = ceil_div(M, t.mt) * tiles_n;
  const int64_t on_cu = ceil_div(splits * ceil_div(tiles, 8), std::max(cus / 8, 1));
  const int64_t per = ceil_div(K / kGroup, splits);
  const float x_mb = 2e-6f * M * K;
  float us = t.fixed + t.per_wg * (on_cu - 1) + t.per_mb * weight_mb(N, K, int4 && !t.dense) +
             t.per_x_mb * tiles_n * x_mb +
             per * ((on_cu / t.per_cu) * t.load[t.per_cu] + t.load[on_cu % t.per_cu]);
  if (splits > 1) us += t.split + t.per_split * splits;
  if (x_mb > 32) us = std::max(us, 0.13f * tiles_n * x_mb);  // X read past the L2s, at 7.7 TB/s
  if (t.mt == 256) us *= 0.98f;                              // ties go to the largest tile
  if (int4 && t.dense) us += 2.5f + 0.62e-6f * N * K;        // unpacking the weight first
  return us;
}

// The same for gemv_kernel (1 to 16 rows): its workgroups on a CU add up, every one reads the M
// rows of X, and each pass over its waves' chunks (24 groups packed, 12 fp16) costs a latency.
inline float gemv_cost(int64_t M, int64_t N, int64_t K, bool int4, int cus) {
  const int64_t groups = K / kGroup;
  const float load = (float)ceil_div(ceil_div(N, 16), cus);
  const float passes = (float)ceil_div(groups, int4 ? 24 : 12) - 1, mb = weight_mb(N, K, int4);
  // 3% off: within the model's error the simpler kernel, with no workspace
  return 0.97f * (int4 ? 3.8448f + 1.2024f * (load - 1) + groups * (0.0204f + 0.0026f * load * M) + 0.1016f * mb +
                         passes * (1.3374f + 1.1724f * (load - 1)) + 0.0725f * load * M
                       : 4.0113f + 1.2468f * (load - 1) + groups * (0.0168f + 0.0037f * load * M) + 0.0595f * mb +
                         passes * (1.4026f + 1.3258f * (load - 1)) + 0.0341f * load * M);
}

// fp32 partial sums of a tiled plan, bytes
inline int64_t partial_bytes(int64_t M, int64_t N, const Plan& pl) {
  return pl.splits <= 1 ? 0 : pl.splits * ceil_div(M, pl.mt) * pl.mt * ceil_div(N, pl.nt) * pl.nt * 4;
}

// The cheapest plan whose partials take at most `room` bytes.  Up to kFusedNormM rows gemv_kernel
// where it takes the norm in, and for fp16 weights so wide that it fills every CU four times (the
// model misses whole rounds of it: 2 rows x 16384 columns, K 11008 72.5 us, 81.9 tiled).
inline Plan choose_plan(int64_t M, int64_t N, int64_t K, bool int4, bool norm, int cus,
                        int64_t room) {
  const int64_t groups = K / kGroup;
  // the partials of a call that large stay within the unpacked weight's bytes
  if (M >= kDenseMinM) room = std::min(room, N * K * 2);
  Plan best{true, false, 16, 16, 1};
  if (M <= kFusedNormM && (norm || (!int4 && ceil_div(N, 16) >= 4 * (int64_t)cus))) return best;
  float best_us = M <= kGemvMaxM ? gemv_cost(M, N, K, int4, cus) : 1e30f;
  const TileCost* costs = int4 ? kPackedTiles : kHalfTiles;
  const int n = int4 ? (int)(sizeof(kPackedTiles) / sizeof(TileCost))
                     : (int)(sizeof(kHalfTiles) / sizeof(TileCost));
  for (int c = 0; c < n; ++c) {
    const TileCost& t = costs[c];
    if (int4 && t.dense && M < kDenseMinM) continue;
    const int64_t tiles = ceil_div(M, t.mt) * ceil_div(N, t.nt);
    // only tiles that the rows fill at least half, and small ones while they are few (others
    // were not timed)
    if ((t.mt > 32 && t.mt >= 2 * M) || (t.mt < 128 && M > 8 * t.mt && tiles > 1024)) continue;
    if (tiles > kMaxTiles) continue;
    const bool may_split = t.split > 0 && tiles <= kMaxSplitTiles;
    for (int64_t s = 1; s <= kMaxSplits && s <= groups; ++s) {
      if (s > 1 && (!may_split || tiles * s > 5 * (int64_t)cus)) break;
      const int64_t per = ceil_div(groups, s), splits = ceil_div(groups, per);
      if (splits != s) continue;  // a smaller count with the same groups per split
      const Plan pl{false, t.dense, t.mt, t.nt, (int)splits};
      if (partial_bytes(M, N, pl) > room) break;
      const float us = tile_cost(t, M, N, K, splits, int4, cus);
      if (us < best_us) {
        best_us = us;
        best = pl;
      }
    }
  }
  return best;
}

// choose_plan, remembered per thread for the last few sizes (it weighs some 60 plans).
inline Plan plan(int64_t M, int64_t N, int64_t K, bool int4, bool norm, int cus) {
  struct Entry {
    int64_t M, N, K;
    int form;
    Plan pl;
  };
  static thread_local Entry memo[64] = {};
  const int form = 4 * cus + 2 * norm + int4;
  Entry& e = memo[(M * 31 + N * 7 + K / kGroup * 3 + form) & 63];
  if (e.M != M || e.N != N || e.K != K || e.form != form)
    e = Entry{M, N, K, form, choose_plan(M, N, K, int4, norm, cus, INT64_MAX)};
  return e.pl;
}

// Bytes of partials without which a call of 17 to 128 rows is refused; with this much, or what
// its plan takes if that is less, it runs (on a plan that fits).  Most of these calls need none:
// the bound is what a split into about two workgroups per CU, kept below the weight's bytes,
// takes (packed weights up to 64 rows: one workgroup per CU, at most eight groups each).
inline int64_t least_partials(int64_t M, int64_t N, int64_t K, bool int4, int cus) {
  const int64_t groups = K / kGroup, tiles = ceil_div(N, kNTile);
  const bool few = int4 && M <= 64;
  int64_t s = 1;
  if (few)
    s = std::max(ceil_div(groups, 8), std::min(groups, cus / tiles));
  else if (tiles < 256)
    s = std::min({ceil_div(512, tiles), std::max<int64_t>(1, K / (16 * M)), groups});
  s = ceil_div(groups, ceil_div(groups, s));
  if (s == 1) return 0;
  return 4 * s * (few ? tiles * kNTile * (M <= 32 ? 32 : 64) : M * N);
}

}  // namespace gemm
}  // namespace fi

namespace {

using fi::half_t;
using fi::gemm::dequantize_kernel;

// Shared validation for the linear-layer entry points; FI_OK when the operands are usable.
int check_linear(const char* fn, const void* x, int64_t x_stride, int64_t M, int64_t K,
                 const void* w, int64_t w_stride, const void* scales, int64_t s_stride,
                 int64_t N, int64_t groupsize, const void* out, int64_t out_stride) {
  using namespace fi;
  using namespace fi::gemm;
  if (M < 0 || N < 0 || K < 0) {
    set_error("%s: negative size", fn);
    return FI_ERR_INVALID;
  }
  if (M == 0 || N == 0) return FI_OK;
  const bool int4 = scales != nullptr;
  if (int4 && groupsize != kGroup) {
    set_error("%s: groupsize %lld not supported (only %d)", fn, (long long)groupsize, kGroup);
    return FI_ERR_UNSUPPORTED;
  }
  if (K == 0 || K % kGroup) {
    set_error("%s: K %lld must be a positive multiple of %d", fn, (long long)K, kGroup);
    return FI_ERR_UNSUPPORTED;
  }
  if (M >= (1ll << 30) || N >= (1ll << 30) || K >= (1ll << 30)) {
    set_error("%s: sizes too large", fn);
    return FI_ERR_UNSUPPORTED;
  }
  if (!x || !w || !out) {
    set_error("%s: null pointer", fn);
    return FI_ERR_INVALID;
  }
  const bool x_ok = ((uintptr_t)x & 15) == 0 && x_stride % 8 == 0 && x_stride >= K;
  const bool w_ok = int4 ? (((uintptr_t)w & 15) == 0 && w_stride % 16 == 0 && w_stride >= K / 2 &&
                            ((uintptr_t)scales & 1) == 0 && s_stride >= K / kGroup)
                         : (((uintptr_t)w & 15) == 0 && w_stride % 8 == 0 && w_stride >= K);
  if (!x_ok || !w_ok || ((uintptr_t)out & 1) || out_stride < N) {
    set_error("%s: rows must be 16-byte aligned and strides cover the rows "
              "(x_stride %lld, w_stride %lld, out_stride %lld)", fn, (long long)x_stride,
              (long long)w_stride, (long long)out_stride);
    return FI_ERR_INVALID;
  }
  return FI_OK;
}

// mid_gemm_kernel and tile_gemm_kernel address the tile's rows of X (and tile_gemm_kernel those
// of W) with 32-bit buffer offsets.
bool spans_ok(const fi::gemm::Params& p, const fi::gemm::Plan& pl) {
  const int64_t x_span = ((pl.mt - 1) * p.x_stride + p.K) * 2;
  const int64_t w_span = pl.dense ? ((pl.nt - 1) * p.w_stride + p.K) * 2 : 0;
  return x_span < 0x7ffffff0 && w_span < 0x7ffffff0;
}

template <typename Kernel, typename Reduce>
void launch_tiles(Kernel kernel, Reduce reduce, const fi::gemm::Params& p, int64_t tile_floats,
                  hipStream_t st) {
  const dim3 grid((unsigned)(8 * p.ksplit * ((p.tiles + 7) / 8)));
  hipLaunchKernelGGL(kernel, grid, dim3(fi::gemm::kThreads), 0, st, p);
  if (p.ksplit > 1 && !p.counters) {
    const int64_t threads = p.tiles * tile_floats / 4;
    hipLaunchKernelGGL(reduce, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p);
  }
}

template <int TM, int NB>
void launch_mid(const fi::gemm::Params& p, hipStream_t st) {
  using namespace fi::gemm;
  launch_tiles(mid_gemm_kernel<TM, NB>, mid_reduce_kernel<TM, NB>, p, TM * 64 * NB, st);
}

template <int BM, int BN, int S>
void launch_tile_gemm(fi::gemm::Params p, hipStream_t st) {
  using namespace fi::gemm;
  p.band = BM == 8 && BN == 8 && p.tiles_m % 8 == 0 ? p.tiles_m / 8 : 0;
  launch_tiles(tile_gemm_kernel<BM, BN, S>, tile_reduce_kernel<BM, BN>, p, 1024 * BM * BN, st);
}

// A tiled plan's launch.  Without arrival counters (a stream past the per-device sets, a device
// whose dispatch does not group block ids by XCD, a first call under graph capture) the
// workgroups only store their partials and a second launch adds them, in the same order.
void launch_plan(fi::gemm::Params p, const fi::gemm::Plan& pl, void* workspace, hipStream_t st) {
  using namespace fi::gemm;
  p.groups_per_split = (int)ceil_div(p.K / kGroup, pl.splits);
  p.partial = (float*)workspace;
  p.tiles_m = (int)ceil_div(p.M, pl.mt);
  p.tiles = p.tiles_m * (int)ceil_div(p.N, pl.nt);
  p.ksplit = pl.splits;
  if (pl.splits > 1)
    p.counters = fi::xcd_counters(st, (p.tiles + 7) / 8, &p.counter_stride);
  p.vec_out = ((uintptr_t)p.out & 15) == 0 && p.out_stride % 8 == 0 && p.N % 8 == 0;
  const int tile = pl.mt * 1000 + pl.nt;
  if (pl.dense) {
    switch (tile) {
      case 32064: launch_tile_gemm<1, 2, 5>(p, st); break;
      case 64064: launch_tile_gemm<2, 2, 4>(p, st); break;
      case 64128: launch_tile_gemm<2, 4, 3>(p, st); break;
      case 128064: launch_tile_gemm<4, 2, 3>(p, st); break;
      case 128128: launch_tile_gemm<4, 4, 2>(p, st); break;
      default: launch_tile_gemm<8, 8, 2>(p, st); break;
    }
    return;
  }
  switch (tile) {
    case 16064: launch_mid<16, 1>(p, st); break;
    case 32064: launch_mid<32, 1>(p, st); break;
    case 64064: launch_mid<64, 1>(p, st); break;
    case 64128: launch_mid<64, 2>(p, st); break;
    case 128064: launch_mid<128, 1>(p, st); break;
    default: launch_mid<128, 2>(p, st); break;
  }
}

void launch_rmsnorm(const half_t* x, int64_t x_stride, int64_t M, int64_t K, const half_t* w,
                    float eps, half_t* out, int64_t out_stride, hipStream_t st) {
  using namespace fi::gemm;
  const int64_t wave_rows = K <= 2048 ? kWaveRows : K < 2816 ? kMoreRows : kManyRows;
  if (K <= kRowParts * 2048 && M < wave_rows)
    hipLaunchKernelGGL(rmsnorm_row_kernel, dim3((unsigned)M), dim3(256), 0, st, x, x_stride, (int)K, w,
                       eps, out, out_stride);
  else
    hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, st, x, x_stride,
                       (int)M, (int)K, w, eps, out, out_stride);
}

// gemv_kernel; `norm`: with the RMSNorm fused into it.  Packed weights: eight waves (two per SIMD
// hide the unpacking's VALU latency), except with a row of the norm per wave, whose registers
// allow only one such workgroup per CU.
void launch_gemv(const fi::gemm::Params& p, bool int4, bool norm, hipStream_t st) {
  using namespace fi::gemm;
  const dim3 grid((unsigned)((p.N + 15) / 16), (unsigned)((p.M + 15) / 16), 1);
  const size_t lds = norm ? (size_t)p.M * p.K * sizeof(half_t) : 0;
  const dim3 four(256), eight(512);
  if (!norm && int4)
    hipLaunchKernelGGL((gemv_kernel<true, 3, 0, 8>), grid, eight, lds, st, p);
  else if (!norm)
    hipLaunchKernelGGL((gemv_kernel<false, 3, 0, 4>), grid, four, lds, st, p);
  else if (!int4)
    hipLaunchKernelGGL((gemv_kernel<false, 3, 4, 4>), grid, four, lds, st, p);
  else if (p.M == 1)
    hipLaunchKernelGGL((gemv_kernel<true, 3, 1, 8>), grid, eight, lds, st, p);
  else if (p.M == 2 && p.K > kShortRow)
    hipLaunchKernelGGL((gemv_kernel<true, 3, 2, 8>), grid, eight, lds, st, p);
  else
    hipLaunchKernelGGL((gemv_kernel<true, 6, 4, 4>), grid, four, lds, st, p);
}

// gemm_kernel: calls of 17 to 128 rows whose rows lie too far apart for 32-bit offsets, with
// the K splits (and workspace) of their plan.
void launch_far_rows(fi::gemm::Params p, bool int4, int splits, void* workspace, hipStream_t st) {
  using namespace fi::gemm;
  p.partial = splits > 1 ? (float*)workspace : nullptr;
  p.groups_per_split = (int)ceil_div(p.K / kGroup, splits);
  const dim3 grid((unsigned)ceil_div(p.N, kNTile), (unsigned)ceil_div(p.M, 32), (unsigned)splits);
  if (int4)
    hipLaunchKernelGGL((gemm_kernel<32, true>), grid, dim3(kThreads), 0, st, p);
  else
    hipLaunchKernelGGL((gemm_kernel<32, false>), grid, dim3(kThreads), 0, st, p);
  if (splits == 1) return;
  const int64_t total = (int64_t)p.M * p.N;
  const int64_t blocks = std::min<int64_t>((total + 255) / 256, 4096);
  hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                     (const float*)workspace, splits, p.M, p.N, p.out, p.out_stride);
}

fi::gemm::Params make_params(const void* x, int64_t x_stride, int64_t M, int64_t K,
                             const void* w, int64_t w_stride, const void* scales,
                             int64_t s_stride, int64_t N, void* out, int64_t out_stride) {
  fi::gemm::Params p;
  p.x = (const half_t*)x;
  p.x_stride = x_stride;
  p.M = (int)M;
  p.K = (int)K;
  p.N = (int)N;
  p.w = (const uint8_t*)w;
  p.w_stride = w_stride;
  p.scales = (const half_t*)scales;
  p.s_stride = s_stride;
  p.out = (half_t*)out;
  p.out_stride = out_stride;
  p.partial = nullptr;
  p.groups_per_split = 0;
  p.norm_w = nullptr;
  p.eps = 0.f;
  p.tiles = 0;
  p.tiles_m = 1;
  p.ksplit = 1;
  p.counters = nullptr;
  p.counter_stride = 0;
  p.band = 0;
  p.vec_out = 0;
  return p;
}

// The norm is fused into the decode kernel for a few rows (each workgroup normalizes them
// into LDS once); otherwise a separate RMSNorm pass writes the normalized rows into the
// workspace first (every column tile would re-read and re-normalize its rows).
bool fuse_norm(int64_t M, int64_t K, const fi::gemm::Plan& pl) {
  // up to 4 rows (measured: the fused call is faster than norm pass + GEMM there); the
  // decode kernel keeps its normalized rows in LDS: at most 64 KB of them
  return pl.gemv && M <= fi::gemm::kFusedNormM && M * K * 2 <= 65536;
}

size_t round256(int64_t n) { return (size_t)((n + 255) / 256 * 256); }

size_t norm_rows_bytes(int64_t M, int64_t K) { return round256(M * K * 2); }

// Workspace layout of a call: [normalized rows (separate norm pass)] [the unpacked weight
// (dense plan, packed weights) or the fp32 partials (split K)], each 256-byte aligned.
struct Layout {
  size_t rows, rest, total;
};

Layout layout(int64_t M, int64_t N, int64_t K, const fi::gemm::Plan& pl, bool int4, bool norm) {
  using namespace fi::gemm;
  Layout l;
  l.rows = norm && !fuse_norm(M, K, pl) ? norm_rows_bytes(M, K) : 0;
  l.rest = pl.gemv ? 0
           : pl.dense && int4 ? round256(N * K * 2)
                              : round256(partial_bytes(M, N, pl));
  l.total = l.rows + l.rest;
  return l;
}

// What the size queries report: the larger of the packed and the fp16 weight forms; from
// kDenseMinM rows, room for the unpacked weight (which also holds any plan's partials).
size_t workspace_bytes_for(int64_t M, int64_t N, int64_t K, bool norm) {
  using namespace fi::gemm;
  const int cus = fi::device_cu_count(nullptr);
  const Layout packed = layout(M, N, K, plan(M, N, K, true, norm, cus), true, norm);
  const Layout half = layout(M, N, K, plan(M, N, K, false, norm, cus), false, norm);
  if (M >= kDenseMinM) return packed.rows + round256(N * K * 2);
  return std::max(packed.total, half.total);
}

// One linear-layer call on any path; norm_w non-null applies RMSNorm to X first.
int run_linear(const char* fn, const void* x, int64_t x_stride, int64_t M, int64_t K,
               const void* norm_w, float eps, const void* w, int64_t w_stride,
               const void* scales, int64_t s_stride, int64_t N, void* out, int64_t out_stride,
               void* workspace, size_t workspace_bytes, hipStream_t st) {
  using namespace fi;
  using namespace fi::gemm;
  const bool int4 = scales != nullptr;
  const bool norm = norm_w != nullptr;
  const int cus = device_cu_count(st);
  if (!workspace || ((uintptr_t)workspace & 255)) workspace_bytes = 0;
  Plan pl = plan(M, N, K, int4, norm, cus);
  Layout l = layout(M, N, K, pl, int4, norm);
  // A call without room for its plan's partials runs on a plan that fits: up to kGemvMaxM rows
  // gemv_kernel, from there the cheapest with what there is.  Packed weights from kDenseMinM
  // rows always need the size queried, 17 to 128 rows least_partials.
  size_t need = l.total;
  if (M >= kDenseMinM && int4) {
    need = l.rows + round256(N * K * 2);
  } else if (workspace_bytes < l.total) {
    if (M > kGemvMaxM && M < kDenseMinM)
      need = std::min(l.total, l.rows + round256(least_partials(M, N, K, int4, cus)));
    else
      need = l.rows;
    if (workspace_bytes >= need) {
      pl = M <= kGemvMaxM ? Plan{true, false, 16, 16, 1}
                          : choose_plan(M, N, K, int4, norm, cus, (int64_t)(workspace_bytes - l.rows));
      l = layout(M, N, K, pl, int4, norm);
    }
  }
  if (workspace_bytes < need) {
    set_error("%s: workspace of %zu bytes (256-byte aligned) needed, %zu given", fn, need,
              workspace_bytes);
    return FI_ERR_WORKSPACE;
  }
  // from kDenseMinM rows every plan keeps the limit of the 256-row tiles
  if (M >= kDenseMinM &&
      (255 * std::max(norm ? K : x_stride, int4 ? K : w_stride) + K) * 2 >= 0x7ffffff0) {
    set_error("fi_int4_matmul: 256 rows of X or W span 2^31 bytes or more");
    return FI_ERR_UNSUPPORTED;
  }
  if (pl.gemv && M > kGemvMaxM) {  // no tiled plan: more than kMaxTiles tiles of any shape
    set_error("fi_int4_matmul: too many output tiles");
    return FI_ERR_UNSUPPORTED;
  }
  // the decode kernel addresses a workgroup's 16 X rows through one buffer descriptor whose
  // size must stay below the offset its idle lanes use (0x7ffffff0)
  const bool fused = norm && fuse_norm(M, K, pl);
  const int64_t gemv_x_stride = norm && !fused ? K : x_stride;
  if (M <= kGemvMaxM && (M - 1) * gemv_x_stride * 2 + K * 2 > 0x7ffffff0) {
    set_error("%s: 16 rows of X span 2^31 bytes or more (x_stride %lld)", fn,
              (long long)x_stride);
    return FI_ERR_UNSUPPORTED;
  }
  char* ws = (char*)workspace;
  Params p = make_params(x, x_stride, M, K, w, w_stride, scales, s_stride, N, out, out_stride);
  if (fused) {
    p.norm_w = (const half_t*)norm_w;
    p.eps = eps;
    launch_gemv(p, int4, true, st);
    return check_launch(fn);
  }
  if (norm) {  // separate norm pass into the workspace
    half_t* normed = (half_t*)ws;
    launch_rmsnorm((const half_t*)x, x_stride, M, K, (const half_t*)norm_w, eps, normed, K, st);
    p.x = normed;
    p.x_stride = K;
  }
  if (pl.gemv) {
    launch_gemv(p, int4, false, st);
    return check_launch(fn);
  }
  if (pl.dense && int4) {  // unpack the weight into the workspace
    half_t* deq = (half_t*)(ws + l.rows);
    const int64_t items = N * (K / 8);
    const int64_t blocks = std::min<int64_t>((items + 255) / 256, 65536);
    hipLaunchKernelGGL(dequantize_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                       (const uint8_t*)w, w_stride, (const half_t*)scales, s_stride, (int)N,
                       (int)K, kGroup, deq, K);
    p.w = (const uint8_t*)deq;
    p.w_stride = K;
  }
  if (spans_ok(p, pl))
    launch_plan(p, pl, ws + l.rows, st);
  else if (M <= kGemvMaxM)
    launch_gemv(p, int4, false, st);
  else
    launch_far_rows(p, int4, pl.splits, ws + l.rows, st);
  return check_launch(fn);
}

}  // namespace

extern "C" int fi_selftest_linear_plan(int64_t M, int64_t N, int64_t K, int packed, int norm,
                                       int32_t* plan) {
  using namespace fi;
  clear_error();
  if (M <= 0 || N <= 0 || K <= 0 || K % gemm::kGroup || M >= (1ll << 30) || N >= (1ll << 30) ||
      K >= (1ll << 30) || !plan) {
    set_error("fi_selftest_linear_plan: sizes must be positive and K a multiple of %d", gemm::kGroup);
    return FI_ERR_INVALID;
  }
  const gemm::Plan pl = gemm::plan(M, N, K, packed != 0, norm != 0, device_cu_count(nullptr));
  plan[0] = pl.gemv ? 0 : pl.dense ? 2 : 1;
  plan[1] = pl.mt;
  plan[2] = pl.nt;
  plan[3] = pl.splits;
  return FI_OK;
}

extern "C" size_t fi_int4_matmul_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % fi::gemm::kGroup) return 0;
  return workspace_bytes_for(M, N, K, false);
}

extern "C" int fi_int4_matmul(const void* x, int64_t x_stride, int64_t M, int64_t K,
                              const void* w, int64_t w_stride, const void* scales,
                              int64_t s_stride, int64_t N, int64_t groupsize, void* out,
                              int64_t out_stride, void* workspace, size_t workspace_bytes,
                              void* stream) {
  using namespace fi;
  clear_error();
  int rc = check_linear("fi_int4_matmul", x, x_stride, M, K, w, w_stride, scales, s_stride, N,
                        groupsize, out, out_stride);
  if (rc != FI_OK || M == 0 || N == 0) return rc;
  return run_linear("fi_int4_matmul", x, x_stride, M, K, nullptr, 0.f, w, w_stride, scales,
                    s_stride, N, out, out_stride, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" size_t fi_rmsnorm_int4_matmul_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % fi::gemm::kGroup) return 0;
  return workspace_bytes_for(M, N, K, true);
}

extern "C" int fi_rmsnorm_int4_matmul(const void* x, int64_t x_stride, int64_t M, int64_t K,
                                      const void* norm_weight, float eps, const void* w,
                                      int64_t w_stride, const void* scales, int64_t s_stride,
                                      int64_t N, int64_t groupsize, void* out,
                                      int64_t out_stride, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  using namespace fi;
  clear_error();
  int rc = check_linear("fi_rmsnorm_int4_matmul", x, x_stride, M, K, w, w_stride, scales,
                        s_stride, N, groupsize, out, out_stride);
  if (rc != FI_OK || M == 0 || N == 0) return rc;
  if (!norm_weight || ((uintptr_t)norm_weight & 15)) {
    set_error("fi_rmsnorm_int4_matmul: norm weight missing or not 16-byte aligned");
    return FI_ERR_INVALID;
  }
  return run_linear("fi_rmsnorm_int4_matmul", x, x_stride, M, K, norm_weight, eps, w, w_stride,
                    scales, s_stride, N, out, out_stride, workspace, workspace_bytes,
                    (hipStream_t)stream);
}

extern "C" int fi_rmsnorm(const void* x, int64_t x_stride, int64_t M, int64_t hidden,
                          const void* weight, float eps, void* out, int64_t out_stride,
                          void* stream) {
  using namespace fi;
  using namespace fi::gemm;
  clear_error();
  if (M < 0 || hidden < 0 || hidden >= (1ll << 30) || M >= (1ll << 30)) {
    set_error("fi_rmsnorm: invalid sizes M %lld hidden %lld", (long long)M, (long long)hidden);
    return FI_ERR_INVALID;
  }
  if (M == 0 || hidden == 0) return FI_OK;
  if (hidden % 8) {
    set_error("fi_rmsnorm: hidden %lld must be a multiple of 8", (long long)hidden);
    return FI_ERR_UNSUPPORTED;
  }
  if (!x || !weight || !out) {
    set_error("fi_rmsnorm: null pointer");
    return FI_ERR_INVALID;
  }
  if (((uintptr_t)x & 15) || ((uintptr_t)weight & 15) || ((uintptr_t)out & 15) ||
      x_stride % 8 || out_stride % 8 || x_stride < hidden || out_stride < hidden) {
    set_error("fi_rmsnorm: rows must be 16-byte aligned and strides cover the rows");
    return FI_ERR_INVALID;
  }
  launch_rmsnorm((const half_t*)x, x_stride, M, hidden, (const half_t*)weight, eps, (half_t*)out,
                 out_stride, (hipStream_t)stream);
  return check_launch("fi_rmsnorm");
}

extern "C" int fi_int4_quantize(const void* w, int64_t w_stride, int64_t N, int64_t K,
                                int64_t groupsize, void* packed, int64_t p_stride,
                                void* scales, int64_t s_stride, void* stream) {
  using namespace fi;
  using namespace fi::gemm;
  clear_error();
  if (groupsize < 8 || groupsize > 512 || (groupsize & (groupsize - 1))) {
    set_error("fi_int4_quantize: groupsize %lld not supported (a power of two from 8 to 512)",
              (long long)groupsize);
    return FI_ERR_UNSUPPORTED;
  }
  if (N < 0 || K < 0 || K % groupsize || N >= (1ll << 30) || K >= (1ll << 30)) {
    set_error("fi_int4_quantize: invalid sizes N %lld K %lld", (long long)N, (long long)K);
    return FI_ERR_INVALID;
  }
  if (N == 0 || K == 0) return FI_OK;
  if (!w || !packed || !scales) {
    set_error("fi_int4_quantize: null pointer");
    return FI_ERR_INVALID;
  }
  if (((uintptr_t)w & 15) || w_stride % 8 || w_stride < K || ((uintptr_t)packed & 3) ||
      p_stride % 4 || p_stride < K / 2 || ((uintptr_t)scales & 1) || s_stride < K / groupsize) {
    set_error("fi_int4_quantize: misaligned rows or short strides");
    return FI_ERR_INVALID;
  }
  const int64_t lanes = N * K / 8;  // gs / 8 per group
  const int64_t blocks = std::min<int64_t>((lanes + 255) / 256, 65536);
  hipLaunchKernelGGL(quantize_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const half_t*)w, w_stride, (int)N, (int)K, (int)groupsize,
                     (uint8_t*)packed, p_stride,
                     (half_t*)scales, s_stride);
  return check_launch("fi_int4_quantize");
}

extern "C" int fi_int4_dequantize(const void* packed, int64_t p_stride, const void* scales,
                                  int64_t s_stride, int64_t N, int64_t K, int64_t groupsize,
                                  void* w, int64_t w_stride, void* stream) {
  using namespace fi;
  using namespace fi::gemm;
  clear_error();
  if (groupsize < 8 || groupsize > 512 || (groupsize & (groupsize - 1))) {
    set_error("fi_int4_dequantize: groupsize %lld not supported (a power of two from 8 to 512)",
              (long long)groupsize);
    return FI_ERR_UNSUPPORTED;
  }
  if (N < 0 || K < 0 || K % groupsize || N >= (1ll << 30) || K >= (1ll << 30)) {
    set_error("fi_int4_dequantize: invalid sizes N %lld K %lld", (long long)N, (long long)K);
    return FI_ERR_INVALID;
  }
  if (N == 0 || K == 0) return FI_OK;
  if (!w || !packed || !scales) {
    set_error("fi_int4_dequantize: null pointer");
    return FI_ERR_INVALID;
  }
  if (((uintptr_t)w & 15) || w_stride % 8 || w_stride < K || ((uintptr_t)packed & 3) ||
      p_stride % 4 || p_stride < K / 2 || ((uintptr_t)scales & 1) || s_stride < K / groupsize) {
    set_error("fi_int4_dequantize: misaligned rows or short strides");
    return FI_ERR_INVALID;
  }
  const int64_t items = N * (K / 8);
  const int64_t blocks = std::min<int64_t>((items + 255) / 256, 65536);
  hipLaunchKernelGGL(dequantize_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     (hipStream_t)stream, (const uint8_t*)packed, p_stride,
                     (const half_t*)scales, s_stride, (int)N, (int)K, (int)groupsize,
                     (half_t*)w, w_stride);
  return check_launch("fi_int4_dequantize");
}
