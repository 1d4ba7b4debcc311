// sbq_quant.hip - weight quantization, packing and activation statistics.
//
//   quantize_per_channel  (spikingbrain_cpu/quant.py:25-29)
//   repack / unpack / colsum (the device-side form of the buffers built by
//                            quant.py:33-39 and the prepack of quant.py:57-61)
//   activation min/max partials (first step of fbgemm's dynamic quantization,
//                                reached from quant.py:65)
#include "sbq_common.h"
#include "sbq_launch.h"

namespace sbq {

// ---------------------------------------------------------------------------
// Weights: quantize_per_channel, the packed tiles and the column sums
// ---------------------------------------------------------------------------
// 16 consecutive values of a weight row as loaded (WT: a source dtype, or
// XT_S8 for rows that are int8 already).
template <int WT>
struct WRaw {
  static constexpr int ES = WT == XT_S8 ? 1 : (WT == XT_F32 ? 4 : 2);
  u32x4 d[ES];

  // columns k0 .. k0 + 15 of the row at p (nullptr: a row of padding); columns
  // >= K are 0.  Rows may start at any address: whole chunks are 16-byte loads
  // of whatever alignment (the GPU splits them), the row's last chunk goes by
  // elements.
  __device__ __forceinline__ void load(const uint8_t* p, int64_t k0, int64_t K) {
    typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
    if (p && k0 + 16 <= K) {
#pragma unroll
      for (int i = 0; i < ES; ++i) d[i] = *(const u32x4_any*)(p + k0 * ES + 16 * i);
      return;
    }
    uint32_t w[4 * ES];
#pragma unroll
    for (int i = 0; i < 4 * ES; ++i) w[i] = 0u;
    if (p && k0 < K) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int64_t k = k0 + j < K ? k0 + j : K - 1;
        uint32_t b;
        if constexpr (ES == 4) b = *(const uint32_t*)(p + k * 4);
        else if constexpr (ES == 2) b = *(const uint16_t*)(p + k * 2);
        else b = p[k];
        if (k0 + j < K) w[j * ES / 4] |= b << (8 * (j * ES % 4));
      }
    }
#pragma unroll
    for (int i = 0; i < ES; ++i) d[i] = (u32x4){w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]};
  }
  __device__ __forceinline__ float get(int j) const {
    const uint32_t word = d[j * ES / 16][j * ES / 4 % 4];  // (a bit_cast of the element itself reads element 0)
    if constexpr (WT == XT_F32) return __uint_as_float(word);
    else if constexpr (WT == XT_F16) return (float)__builtin_bit_cast(f16x2, word)[j & 1];
    else return __uint_as_float(j & 1 ? word & 0xffff0000u : word << 16);
  }
};

// clamp(rint(v / s), -127, 127) of 16 values as bytes.  The division is IEEE
// (about ten instructions); nearly always its rounded result is that of
// t = v * inv, inv = fp32(1 / s): |v| <= 127 s, so t is within 2.3e-5 of the
// fp32 quotient (1.5 units of 2^-24 each, times 127) and both round alike
// unless t is that close to a half.  Rounding by adding 1.5 * 2^23: the low
// byte of the sum is the integer.  A value near a half, an infinity or a NaN
// takes the division, one by one: of bf16 values about one in 400 is half its
// row's maximum (63.5), so most wavefronts hold one (dividing the whole chunk then
// took 999 x 1001 10.7 us, one wave per row 6.4).
template <int WT>
__device__ __forceinline__ u32x4 quant_w16(const WRaw<WT>& raw, float s, float inv) {
  constexpr float kMagic = 12582912.0f;
  uint32_t m[16];
  uint32_t unsure = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float t = raw.get(j) * inv, r = t + kMagic;
    unsure |= __builtin_fabsf(t - (r - kMagic)) < 0.49997f ? 0u : 1u << j;
    m[j] = __float_as_uint(r);
  }
  if (unsure) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (unsure & (1u << j)) {
        const float t = __builtin_rintf(raw.get(j) / s);
        m[j] = (uint32_t)(int)fminf(fmaxf(t, -127.0f), 127.0f);
      }
    }
  }
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = __builtin_amdgcn_perm(m[4 * i + 1], m[4 * i], 0x0c0c0400u) |
           __builtin_amdgcn_perm(m[4 * i + 3], m[4 * i + 2], 0x04000c0cu);
  return o;
}

// quantize_per_channel of few short rows of 2-byte values, nothing packed: one
// wavefront per row, a division per value.  A few rows leave the kernel below
// few workgroups, its 16-byte loads of rows at odd 2-byte addresses take
// several passes each, and near-half quotients are frequent in bf16.  That
// kernel / this one (bf16, graph): 999 x 1001 8.7 / 6.4 us, 1000 x 2001 13.5 /
// 10.0, 1000 x 1000 7.2 / 6.4; on the other side of the line 4000 x 2001 14.7 /
// 19.3, 2560 x 2501 17.0 / 20.4, 1000 x 2000 9.2 / 9.9, 128 x 2560 10.1 / 11.3.
template <int WT>
__global__ __launch_bounds__(256) void quantize_few_rows_kernel(const void* __restrict__ wv, int64_t N, int64_t K,
                                                                int64_t ldw, int8_t* __restrict__ q, int64_t ldq,
                                                                float* __restrict__ scale) {
  typedef typename XElem<WT>::T T;
  const int lane = threadIdx.x & 63;
  const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const T* row = (const T*)wv + n * ldw;
  float m = 0.0f;
  for (int64_t k = lane; k < K; k += 64) m = fmaxf(m, __builtin_fabsf(XElem<WT>::to_f32(row[k])));
  m = wave_max(m);
  const float s = fmaxf(m, 1e-8f) / 127.0f;
  if (lane == 0) scale[n] = s;
  for (int64_t k = lane; k < K; k += 64) {
    const float t = __builtin_rintf(XElem<WT>::to_f32(row[k]) / s);
    q[n * ldq + k] = (int8_t)(int)fminf(fmaxf(t, -127.0f), 127.0f);
  }
}

// Column sums that several workgroups add to start from zero.
__global__ __launch_bounds__(256) void zero_ints_kernel(int32_t* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = 0;
}

// One workgroup of 8 waves per 16 weight rows: lane (g, r) of wave v takes the
// 16-value chunks of row r at columns 64 kc + 16 g, kc = v, v + 8, ..., the
// chunk that is its 16 bytes of packed tile kc.  With a floating source each
// row's max |w| is reduced (over the lanes of the row, then the waves through
// LDS), scale = max(that, 1e-8) / 127, and the same chunks are quantized; an
// int8 source (repack) is taken as it is.  Writes whatever is asked for: the
// scales, the int8 rows q, the packed tiles (offset binary), the column sums.
// C > 0: the wave's at most C chunks per lane stay in registers between the
// two passes; C = 0: longer rows are read again (from the Infinity Cache).
// HBM bound: one read of w, one write of each output.  Measured (whole call of
// a module's load, eager, against a scalar quantizer, a byte-wise repack and a
// column-sum launch, with the int8 rows written and read twice between them):
// bf16 9728 x 2560 112 -> 22 us, 24576 x 4096 407 -> 65 us (4.7 TB/s),
// 151936 x 2560 1661 -> 213 us (5.5 TB/s); with the int8 rows kept 24 / 89 /
// 300 us; fp32 9728 x 2560 135 -> 24; ragged bf16 9721 x 2555 101 -> 37.  int8
// rows alone, K over several workgroups where there are few row tiles (graph):
// 16 x 65536 44 -> 3.6 us, 64 x 12288 10.3 -> 3.9, 300 x 9728 9.0 -> 4.4, with
// their column sums 44 -> 6.4, 10.5 -> 5.5, 9.2 -> 6.1.  16
// waves per workgroup: 20-45% slower except at K = 9728 (5% faster); holding
// 24 chunks spilled (2560 x 9728: 74 us, re-reading 32).
template <int WT, int C>
__global__ __launch_bounds__(512) void pack_weight_kernel(const uint8_t* __restrict__ w, int64_t N, int64_t K,
                                                          int64_t ldw, float* __restrict__ scale,
                                                          int8_t* __restrict__ q, int64_t ldq,
                                                          uint8_t* __restrict__ packed,
                                                          int32_t* __restrict__ colsum) {
  constexpr int NW = 8, U = 4;
  constexpr bool FP = WT != XT_S8;
  __shared__ float smax[NW][16];
  __shared__ int ssum[NW][16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int64_t nt = blockIdx.x, n = nt * 16 + r, Kc = (K + 63) / 64;
  // int8 rows: K split over gridDim.y workgroups, their column sums added up
  const int64_t share = FP ? Kc : (Kc + gridDim.y - 1) / gridDim.y;
  const int64_t kb = FP ? 0 : blockIdx.y * share, ke = FP ? Kc : (kb + share < Kc ? kb + share : Kc);
  const uint8_t* row = n < N ? w + n * ldw * WRaw<WT>::ES : nullptr;
  WRaw<WT> v[C > 0 ? C : U];
  float s = 0.0f, inv = 0.0f;
  const auto row_max = [&](const WRaw<WT>& x, float m) {
#pragma unroll
    for (int j = 0; j < 16; ++j) m = fmaxf(m, __builtin_fabsf(x.get(j)));
    return m;
  };
  if constexpr (FP) {
    float m = 0.0f;
    if constexpr (C > 0) {
#pragma unroll
      for (int i = 0; i < C; ++i)
        if (wv + i * NW < Kc) v[i].load(row, (wv + i * NW) * 64 + g * 16, K);
#pragma unroll
      for (int i = 0; i < C; ++i)
        if (wv + i * NW < Kc) m = row_max(v[i], m);
    } else {
      for (int64_t kc = wv; kc < Kc; kc += U * NW) {
#pragma unroll
        for (int i = 0; i < U; ++i)
          if (kc + i * NW < Kc) v[i].load(row, (kc + i * NW) * 64 + g * 16, K);
#pragma unroll
        for (int i = 0; i < U; ++i)
          if (kc + i * NW < Kc) m = row_max(v[i], m);
      }
    }
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    if (g == 0) smax[wv][r] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i) m = fmaxf(m, smax[i][r]);
    s = fmaxf(m, 1e-8f) / 127.0f;
    inv = 1.0f / s;
    if (threadIdx.x < 16 && n < N) scale[n] = s;
  }
  int sum = 0;
  const auto emit = [&](int64_t kc, const WRaw<WT>& x) {
    u32x4 b;
    if constexpr (FP) b = quant_w16<WT>(x, s, inv);
    else b = x.d[0];
#pragma unroll
    for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_sdot4((int)b[i], 0x01010101, sum, false);
    if (packed)
      *(u32x4*)(packed + ((nt * Kc + kc) * 64 + lane) * 16) = b ^ (u32x4){0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u};
    const int64_t k0 = kc * 64 + g * 16;
    if (q && n < N) {
      typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
      int8_t* dst = q + n * ldq + k0;
      if (k0 + 16 <= K) {
        *(u32x4_any*)dst = b;
      } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const uint32_t word = b[j / 4];
          if (k0 + j < K) dst[j] = (int8_t)(word >> (8 * (j % 4)));
        }
      }
    }
  };
  if constexpr (C > 0) {
    // the chunks stay as loaded (the compiler would keep the 2-byte values as
    // the floats of the first pass, twice the registers)
#pragma unroll
    for (int i = 0; i < C; ++i)
#pragma unroll
      for (int j = 0; j < WRaw<WT>::ES; ++j) asm("" : "+v"(v[i].d[j]));
#pragma unroll
    for (int i = 0; i < C; ++i)
      if (wv + i * NW < Kc) emit(wv + i * NW, v[i]);
  } else {
    for (int64_t kc = kb + wv; kc < ke; kc += U * NW) {
#pragma unroll
      for (int i = 0; i < U; ++i)
        if (kc + i * NW < ke) v[i].load(row, (kc + i * NW) * 64 + g * 16, K);
#pragma unroll
      for (int i = 0; i < U; ++i)
        if (kc + i * NW < ke) emit(kc + i * NW, v[i]);
    }
  }
  if (colsum) {  // uniform; exact int32: |sum| <= 127 * K
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (g == 0) ssum[wv][r] = sum;
    __syncthreads();
    if (threadIdx.x < 16 && n < N) {
      int t = 0;
#pragma unroll
      for (int i = 0; i < NW; ++i) t += ssum[i][r];
      if (!FP && gridDim.y > 1)
        __hip_atomic_fetch_add(colsum + n, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        colsum[n] = t;
    }
  }
}

// Packed tiles -> int8 rows: one 16-byte lane slot per thread, stored at
// whatever alignment the row has.
__global__ __launch_bounds__(256) void unpack_kernel(const uint8_t* __restrict__ packed, int64_t N, int64_t K,
                                                     int64_t Kc, int64_t nslots, int8_t* __restrict__ q, int64_t ldq) {
  typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
  const int64_t slot = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (slot >= nslots) return;
  const int lane = (int)(slot & 63);
  const int64_t tile = slot >> 6, nt = tile / Kc, kc = tile - nt * Kc;
  const int64_t n = nt * 16 + (lane & 15), k0 = kc * 64 + (lane >> 4) * 16;
  if (n >= N || k0 >= K) return;
  const u32x4 b = *(const u32x4*)(packed + slot * 16) ^ (u32x4){0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u};
  int8_t* dst = q + n * ldq + k0;
  if (k0 + 16 <= K) {
    *(u32x4_any*)dst = b;
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t word = b[j / 4];
      if (k0 + j < K) dst[j] = (int8_t)(word >> (8 * (j % 4)));
    }
  }
}

// The column table of outputs stored as parts, from the parts in the kernel
// arguments (a host copy would wait for everything launched before it).
__global__ __launch_bounds__(256) void parts_fill_kernel(PartsFill f, uint32_t begin4, int32_t* __restrict__ table) {
  const uint32_t i = begin4 + blockIdx.x * 256 + threadIdx.x;
  uint32_t width = 0, word = 0, end = 0;
#pragma unroll
  for (int p = kPartsFill - 1; p >= 0; --p)
    if (p < f.count && i < f.end4[p]) {
      width = f.width[p];
      word = f.word[p];
      end = f.end4[p];
    }
  if (i >= end) return;
  table[2 * i] = (int32_t)width;
  table[2 * i + 1] = (int32_t)word;
}

// Zero the split-K tile counters of the GEMM that follows a pre-pass (the
// pre-pass runs first on the same stream, so the GEMM sees them zeroed).
__device__ __forceinline__ void zero_counters(uint32_t* c, int n) {
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < n; i += blockDim.x) c[i] = 0u;
}

// The block's (min, max) into partials[blockIdx.x]: wave reductions, then
// thread 0 over the waves.
__device__ __forceinline__ void store_block_minmax(float mn, float mx, float2* partials) {
  __shared__ float red[32];
  mn = wave_min(mn);
  mx = wave_max(mx);
  const int wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[2 * wid] = mn;
    red[2 * wid + 1] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < nw; ++w) {
      mn = fminf(mn, red[2 * w]);
      mx = fmaxf(mx, red[2 * w + 1]);
    }
    partials[blockIdx.x] = make_float2(mn, mx);
  }
}

// Dense x (ldx == K, 16-byte aligned, K % 8 == 0): the M*K values are one flat
// array of 8-value chunks (16 bytes of fp16 / bf16, 32 of fp32).  Thread t of
// the grid folds chunks t, t + T, t + 2T, ... (T threads), U loads in flight
// per round with no branch: indexes past the end are clamped to the last
// chunk, whose values are already in the range (min and max are idempotent).
// No division, no per-element guard.
template <int XT, int U>
__global__ __launch_bounds__(1024) void minmax_dense_kernel(const void* __restrict__ xv, int64_t nch,
                                                            float2* __restrict__ partials,
                                                            uint32_t* __restrict__ zero, int nzero) {
  typedef typename XElem<XT>::T T;
  typedef T v8 __attribute__((ext_vector_type(8)));
  zero_counters(zero, nzero);
  const int64_t T_ = (int64_t)gridDim.x * blockDim.x;
  float mn = 0.0f, mx = 0.0f;  // fbgemm's range always holds 0
  for (int64_t c0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c0 < nch; c0 += U * T_) {
    float t[U][8];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int64_t c = min(c0 + i * T_, nch - 1);
      if constexpr (XT == XT_F32) {
        const f32x4 a0 = *(const f32x4*)((const float*)xv + c * 8), a1 = *(const f32x4*)((const float*)xv + c * 8 + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          t[i][j] = a0[j];
          t[i][4 + j] = a1[j];
        }
      } else {
        const v8 a = *(const v8*)((const T*)xv + c * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) t[i][j] = XElem<XT>::to_f32(a[j]);
      }
    }
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        mn = fminf(mn, t[i][j]);
        mx = fmaxf(mx, t[i][j]);
      }
  }
  store_block_minmax(mn, mx, partials);
}

// Per-block (min, max) of x [M, K] with any row stride: thread t of the grid
// covers the 8-value chunks t, t + T, ... (T threads; chunks row by row).
template <int XT>
__global__ __launch_bounds__(1024) void minmax_partial_kernel(const void* __restrict__ xv, int M, int K, int64_t ldx,
                                                              float2* __restrict__ partials, int vec,
                                                              uint32_t* __restrict__ zero, int nzero) {
  zero_counters(zero, nzero);
  const int cpr = (K + 7) / 8;
  const int64_t nch = (int64_t)M * cpr;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  float mn = 0.0f, mx = 0.0f;  // lo <= 0 <= hi after clamping anyway
  auto fold = [&](const float* t, int k0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = k0 + j < K ? t[j] : 0.0f;
      mn = fminf(mn, v);
      mx = fmaxf(mx, v);
    }
  };
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (; c + 3 * stride < nch; c += 4 * stride) {  // four chunks in flight
    float t[4][8];
    int k0[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t ci = c + i * stride;
      const int m = (int)(ci / cpr);
      k0[i] = (int)(ci - (int64_t)m * cpr) * 8;
      load8_f32<XT>(xv, ldx, M, K, m, k0[i], vec, t[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) fold(t[i], k0[i]);
  }
  for (; c < nch; c += stride) {
    const int m = (int)(c / cpr), k0 = (int)(c - (int64_t)m * cpr) * 8;
    float t[8];
    load8_f32<XT>(xv, ldx, M, K, m, k0, vec, t);
    fold(t, k0);
  }
  store_block_minmax(mn, mx, partials);
}

__global__ __launch_bounds__(256) void qparams_kernel(const float2* __restrict__ partials, int nparts,
                                                      float* __restrict__ scale_out, int32_t* __restrict__ zp_out) {
  __shared__ float red[8];
  ActQParams p = block_qparams_from_partials(partials, nparts, red);
  if (threadIdx.x == 0) {
    *scale_out = p.scale;
    *zp_out = p.zp;
  }
}

// ---------------------------------------------------------------------------
// Row argmax of fp32 logits (greedy sampling, engine.py:30-31
// `int(logits.argmax())` over the lm_head output): the first index of the
// largest value, NaN above every number, as torch.argmax.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool arg_better(float v, int i, float bv, int bi) {
  const bool vn = v != v, bn = bv != bv;
  if (vn != bn) return vn;
  if (vn) return i < bi;
  return v > bv || (v == bv && i < bi);
}

__device__ __forceinline__ void arg_take(float v, int i, float& bv, int& bi) {
  if (arg_better(v, i, bv, bi)) {
    bv = v;
    bi = i;
  }
}

// Per-row sums of fp16 activations in fp32 (the offset the prefill GEMM's
// subnormal weight encoding adds: sum_k (q + 128) x_k = sum_k q x_k + 128 * rowsum).
// One wave per row, 16-byte loads (four in flight per lane), two accumulators;
// rows are 16-byte aligned and K % 8 == 0 on this path.
__device__ __forceinline__ void rowsum_acc(u32x4 v, float& s0, float& s1) {
  const uint32_t w0 = v.x, w1 = v.y, w2 = v.z, w3 = v.w;
  const f16x2 one = {1.0f16, 1.0f16};
  s0 = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w0), one, s0, false);
  s1 = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w1), one, s1, false);
  s0 = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w2), one, s0, false);
  s1 = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w3), one, s1, false);
}

__global__ __launch_bounds__(256) void rowsum_f16_kernel(const _Float16* __restrict__ x, int64_t ldx, int M, int K,
                                                         float* __restrict__ out, uint32_t* __restrict__ zero,
                                                         int nzero) {
  zero_counters(zero, nzero);
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const _Float16* p = x + (int64_t)row * ldx;
  float s0 = 0.0f, s1 = 0.0f;
  int k = lane * 8;
  // eight loads in flight (a whole K = 4096 row in one round), then four, then
  // one; the chunks are summed in the same order whichever loop takes them
  for (; k + 7 * 512 < K; k += 8 * 512) {
    u32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = *(const u32x4*)(p + k + j * 512);
#pragma unroll
    for (int j = 0; j < 8; ++j) rowsum_acc(v[j], s0, s1);
  }
  for (; k + 3 * 512 < K; k += 4 * 512) {
    u32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = *(const u32x4*)(p + k + j * 512);
#pragma unroll
    for (int j = 0; j < 4; ++j) rowsum_acc(v[j], s0, s1);
  }
  for (; k < K; k += 512) rowsum_acc(*(const u32x4*)(p + k), s0, s1);
  float s = s0 + s1;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) out[row] = s;
}

// fbgemm's per-tensor activation quantization on its own (the step inside
// quantized::linear_dynamic, quant.py:65, that the int8-dyn GEMMs fuse into
// their pre-pass): the (s_x, zp) of the min/max partials, then
// xq[m,k] = clamp(rint(fma(x[m,k], 1/s_x, zp)), 0, 255) as uint8 [M][ldq],
// the arithmetic of the GEMM path's quantize pass (without its s8 shift).
// One thread per 8 consecutive values of a row; loads clamped to the row,
// stores guarded.
template <int XT>
__global__ __launch_bounds__(256) void act_quant_u8_kernel(const void* __restrict__ x, int64_t ldx, int M, int K,
                                                           bool vec, const float2* __restrict__ partials,
                                                           int nparts, uint8_t* __restrict__ xq, int64_t ldq,
                                                           bool qvec) {
  const int cpr = (K + 7) / 8;
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t cl = min(c, (int64_t)M * cpr - 1);
  const int m = (int)(cl / cpr), k0 = (int)(cl - (int64_t)m * cpr) * 8;
  float t[8];
  load8_f32<XT>(x, ldx, M, K, m, k0, vec, t);
  __shared__ float red[8];
  const ActQParams qp = block_qparams_from_partials(partials, nparts, red);
  if (c >= (int64_t)M * cpr) return;
  uint32_t d[2];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    uint32_t v = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(t[4 * w], qp.inv, qp.zpf), 0, 0u);
    v = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(t[4 * w + 1], qp.inv, qp.zpf), 1, v);
    v = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(t[4 * w + 2], qp.inv, qp.zpf), 2, v);
    d[w] = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(t[4 * w + 3], qp.inv, qp.zpf), 3, v);
  }
  uint8_t* dst = xq + (int64_t)m * ldq + k0;
  if (qvec && k0 + 8 <= K) {
    *(u32x2*)dst = (u32x2){d[0], d[1]};
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 + j < K) dst[j] = (uint8_t)(d[j >> 2] >> (8 * (j & 3)));
  }
}

// Per-token symmetric activation quantization (the opt-in int8-dyn
// granularity): each activation row is quantized exactly as
// quantize_per_channel (spikingbrain_cpu/quant.py:25-29) quantizes a weight
// row: s = max(max_k |x|, 1e-8) / 127 (IEEE division), xq = clamp(rne(x / s),
// -127, 127).  xq rows have Kp bytes; columns K..Kp-1 are written as 0.
template <int XT>
__global__ __launch_bounds__(256) void quantize_rows_sym_kernel(const void* __restrict__ xv, int64_t ldx, int M, int K,
                                                                int Kp, int vec, int8_t* __restrict__ xq,
                                                                float* __restrict__ s_out,
                                                                uint32_t* __restrict__ zero, int nzero) {
  zero_counters(zero, nzero);
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  float amax = 0.0f;
  for (int k = lane * 8; k < K; k += 512) {
    float t[8];
    load8_f32<XT>(xv, ldx, M, K, row, k, vec, t);  // columns >= K read as 0
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, __builtin_fabsf(t[j]));
  }
  amax = wave_max(amax);
  const float sc = fmaxf(amax, 1e-8f) / 127.0f;
  if (lane == 0) s_out[row] = sc;
  int8_t* qrow = xq + (int64_t)row * Kp;
  for (int k = lane * 8; k < Kp; k += 512) {
    float t[8];
    load8_f32<XT>(xv, ldx, M, K, row, k, vec, t);
    uint32_t d[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float v = __builtin_rintf(t[j] / sc);
      v = fminf(fmaxf(v, -127.0f), 127.0f);
      d[j >> 2] |= ((uint32_t)(int)v & 0xffu) << (8 * (j & 3));
    }
    *(u32x2*)(qrow + k) = (u32x2){d[0], d[1]};  // Kp % 64 == 0 and Kp-byte rows: 8-byte aligned
  }
}

// fp32 / bf16 activations -> one power-of-two scaled fp16 plane for the fp16
// prefill GEMM.  Row m is scaled by 2^e (max|x| * 2^e in [2^14, 2^15), an
// exact scaling) and rounded once: plane row m = rn16(x * 2^e).  bf16 values
// (8 significant bits) are exact down to 2^28 below the row maximum; fp32
// values keep 11 bits (relative rounding error <= 2^-11 per value, about 3e-4
// relative L2 on the outputs, inside the 1e-3 weight-only tolerance).
// rowsum[m] = the fp32 sum of the plane's fp16 values; rscale[m] = 2^-e.  One
// wave per row; rows are 16-byte aligned and K % 64 == 0 on this path.  Rows
// of at most 512 * C values are read once, every 8-value chunk of a lane in
// flight together and held in registers for the conversion; longer rows are
// read twice (maximum, then conversion), four chunks in flight.
template <int XT, int C>
__global__ __launch_bounds__(256) void stage_act_kernel(const void* __restrict__ xv, int64_t ldx, int M, int K,
                                                        _Float16* __restrict__ xs, float* __restrict__ rowsum,
                                                        float* __restrict__ rscale, uint32_t* __restrict__ zero,
                                                        int nzero) {
  zero_counters(zero, nzero);
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  typedef typename XElem<XT>::T T;
  const T* xr = (const T*)xv + (int64_t)row * ldx;
  _Float16* out = xs + (int64_t)row * K;
  float mx = 0.0f, s = 0.0f;
  auto convert = [&](const float* t, float sc, int k) {
    f16x8 h;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      h[j] = (_Float16)(t[j] * sc);
      s += (float)h[j];
    }
    *(f16x8*)(out + k) = h;
  };
  int e;
  if (K <= 512 * C) {
    float t[C][8];
#pragma unroll
    for (int c = 0; c < C; ++c)  // clamped: chunks past the row repeat its last chunk, never converted
      load8_f32_vec<XT>(xr + min(lane * 8 + c * 512, K - 8), t[c]);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(t[c][j]));
    e = row_scale_exp(wave_max(mx));
    const float sc = ldexpf(1.0f, e);
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (lane * 8 + c * 512 < K) convert(t[c], sc, lane * 8 + c * 512);
  } else {
    for (int k0 = lane * 8; k0 < K; k0 += 4 * 512) {
      float t[4][8];
#pragma unroll
      for (int c = 0; c < 4; ++c) load8_f32_vec<XT>(xr + min(k0 + c * 512, K - 8), t[c]);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(t[c][j]));
    }
    e = row_scale_exp(wave_max(mx));
    const float sc = ldexpf(1.0f, e);
    for (int k0 = lane * 8; k0 < K; k0 += 4 * 512) {
      float t[4][8];
#pragma unroll
      for (int c = 0; c < 4; ++c) load8_f32_vec<XT>(xr + min(k0 + c * 512, K - 8), t[c]);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (k0 + c * 512 < K) convert(t[c], sc, k0 + c * 512);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) {
    rowsum[row] = s;
    rscale[row] = ldexpf(1.0f, -e);
  }
}

// x as rows of whole K tiles (PLANES 1: a copy in x's dtype; PLANES 2: fp32 as
// bf16 high and remainder planes, [M][2][Kp]); one 8-value chunk per thread,
// loads of whatever alignment, a row's last chunk by elements, padding 0.
template <int XT, int PLANES>
__global__ __launch_bounds__(256) void pad_rows_kernel(const void* __restrict__ xv, int64_t ldx, int64_t nch, int cpr,
                                                       int K, uint8_t* __restrict__ out,
                                                       uint32_t* __restrict__ zero, int nzero) {
  zero_counters(zero, nzero);
  typedef typename XElem<XT>::T T;
  typedef T v4 __attribute__((ext_vector_type(4)));
  typedef T v4_any __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= nch) return;
  const int64_t m = c / cpr;
  const int k0 = (int)(c - m * cpr) * 8;
  const T* p = (const T*)xv + m * ldx + k0;
  v4 v[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (k0 + 4 * h + 4 <= K) {
      v[h] = *(const v4_any*)(p + 4 * h);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[h][j] = k0 + 4 * h + j < K ? p[4 * h + j] : (T)0.0f;
    }
  }
  if constexpr (PLANES == 1) {
    v4* o = (v4*)(out + c * 8 * sizeof(T));
    o[0] = v[0];
    o[1] = v[1];
  } else {
    bf16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      __bf16 a, b;
      split_bf16(XElem<XT>::to_f32(v[j / 4][j % 4]), a, b);
      hi[j] = a;
      lo[j] = b;
    }
    __bf16* o = (__bf16*)out + m * cpr * 16 + k0;
    *(bf16x8*)o = hi;
    *(bf16x8*)(o + cpr * 8) = lo;
  }
}

// One workgroup per row; each thread keeps four independent running bests
// and has sixteen vector loads in flight at a time (a 151936-wide row is
// three rounds of loads).
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const float* __restrict__ y, int N, int64_t ldy,
                                                           int64_t* __restrict__ out, int vec) {
  const float* row = y + (int64_t)blockIdx.x * ldy;
  float bv[4];
  int bi[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    bv[u] = -__builtin_inff();
    bi[u] = 0x7fffffff;
  }
  const int T = blockDim.x, t = threadIdx.x;
  int i0 = 0;
  if (vec) {
    const int n4 = N / 4;
    int c = t;
    for (; c + 15 * T < n4; c += 16 * T) {
      f32x4 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = *(const f32x4*)(row + 4 * (c + u * T));
#pragma unroll
      for (int u = 0; u < 16; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) arg_take(v[u][j], 4 * (c + u * T) + j, bv[u & 3], bi[u & 3]);
    }
    for (; c + 3 * T < n4; c += 4 * T) {
      f32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = *(const f32x4*)(row + 4 * (c + u * T));
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) arg_take(v[u][j], 4 * (c + u * T) + j, bv[u], bi[u]);
    }
    for (; c < n4; c += T) {
      const f32x4 v = *(const f32x4*)(row + 4 * c);
#pragma unroll
      for (int j = 0; j < 4; ++j) arg_take(v[j], 4 * c + j, bv[0], bi[0]);
    }
    i0 = n4 * 4;
  }
  for (int i = i0 + t; i < N; i += T) arg_take(row[i], i, bv[0], bi[0]);
#pragma unroll
  for (int u = 1; u < 4; ++u) arg_take(bv[u], bi[u], bv[0], bi[0]);
  float v = bv[0];
  int i = bi[0];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) arg_take(__shfl_xor(v, o, 64), __shfl_xor(i, o, 64), v, i);
  __shared__ float sv[16];
  __shared__ int si[16];
  if ((t & 63) == 0) {
    sv[t >> 6] = v;
    si[t >> 6] = i;
  }
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < (T >> 6); ++w) arg_take(sv[w], si[w], v, i);
    out[blockIdx.x] = i;
  }
}

// Long rows over many workgroups, with no scratch but the output: out[row]
// holds the row's largest argmax_key (sbq_index.h) until the last launch
// replaces it by the key's column.  One workgroup per row reads 608 KB through
// one CU (V = 151936, one row: 46 us in a HIP graph); these three launches,
// slices of the rows over 64 workgroups: 7.1 us, 8 rows 46 -> 12.4; V = 32000
// 14.9 -> 6.1.
__global__ __launch_bounds__(256) void argmax_clear_kernel(unsigned long long* __restrict__ out, int64_t M) {
  const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (m < M) out[m] = 0ull;  // below every key
}

__global__ __launch_bounds__(256) void argmax_slice_kernel(const float* __restrict__ y, int N, int64_t ldy, int per,
                                                           unsigned long long* __restrict__ out) {
  constexpr int U = 8;
  const int64_t rowi = blockIdx.y;
  const float* row = y + rowi * ldy;
  const int i0 = blockIdx.x * per, i1 = min(i0 + per, N), t = threadIdx.x;
  unsigned long long best = 0;
  for (int b = i0 + t; b < i1; b += U * 256) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = row[min(b + u * 256, i1 - 1)];  // clamped: the slice's last value again
#pragma unroll
    for (int u = 0; u < U; ++u) best = max(best, argmax_key(v[u], min(b + u * 256, i1 - 1)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = max(best, (unsigned long long)__shfl_xor(best, o, 64));
  __shared__ unsigned long long red[4];
  if ((t & 63) == 0) red[t >> 6] = best;
  __syncthreads();
  if (t == 0) {
    best = max(max(red[0], red[1]), max(red[2], red[3]));
    __hip_atomic_fetch_max(out + rowi, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__global__ __launch_bounds__(256) void argmax_index_kernel(unsigned long long* __restrict__ out, int64_t M) {
  const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (m < M) out[m] = (unsigned long long)argmax_key_index(out[m]);
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
int launch_pack_weight(const void* w, int wt, int64_t N, int64_t K, int64_t ldw, float* scale, int8_t* q, int64_t ldq,
                       uint8_t* packed, int32_t* colsum, hipStream_t st) {
  if (!packed && N <= 2048 && (wt == XT_F16 || wt == XT_BF16) && (K <= 1024 || (((uintptr_t)w | ldw * 2) & 2))) {
    const dim3 rows((unsigned)((N + 3) / 4));
    if (wt == XT_F16)
      hipLaunchKernelGGL((quantize_few_rows_kernel<XT_F16>), rows, dim3(256), 0, st, w, N, K, ldw, q, ldq, scale);
    else
      hipLaunchKernelGGL((quantize_few_rows_kernel<XT_BF16>), rows, dim3(256), 0, st, w, N, K, ldw, q, ldq, scale);
    return check_launch();
  }
  const dim3 grid((unsigned)((N + 15) / 16)), block(512);
  const int64_t per = ((K + 63) / 64 + 7) / 8;  // chunks per lane
#define SBQ_PACK(WT_, C_) \
  hipLaunchKernelGGL((pack_weight_kernel<WT_, C_>), grid, block, 0, st, (const uint8_t*)w, N, K, ldw, scale, q, ldq, packed, colsum)
  // held in registers: up to 16 chunks of 2-byte values (199 VGPRs, K <= 8192), 8 of fp32 (175, K <= 4096)
#define SBQ_PACK2(WT_)                          \
  if (per <= 2) SBQ_PACK(WT_, 2);               \
  else if (per <= 5) SBQ_PACK(WT_, 5);          \
  else if (per <= 8) SBQ_PACK(WT_, 8);          \
  else if (per <= 16) SBQ_PACK(WT_, 16);        \
  else SBQ_PACK(WT_, 0)
  switch (wt) {
    case XT_F16: SBQ_PACK2(XT_F16); break;
    case XT_BF16: SBQ_PACK2(XT_BF16); break;
    case XT_F32:
      if (per <= 2) SBQ_PACK(XT_F32, 2);
      else if (per <= 5) SBQ_PACK(XT_F32, 5);
      else if (per <= 8) SBQ_PACK(XT_F32, 8);
      else SBQ_PACK(XT_F32, 0);
      break;
    case XT_S8: {
      // few row tiles of long rows: K over several workgroups, each with a round
      // of K tiles at least; with column sums they start from zero, a launch more
      const int64_t tiles = (N + 15) / 16, share = (512 + tiles - 1) / tiles;
      const unsigned split = tiles >= 256 || (colsum && per <= 8) ? 1u : (unsigned)(share < per ? share : per);
      if (colsum && split > 1)
        hipLaunchKernelGGL(zero_ints_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, st, colsum, N);
      hipLaunchKernelGGL((pack_weight_kernel<XT_S8, 0>), dim3((unsigned)tiles, split), block, 0, st, (const uint8_t*)w,
                         N, K, ldw, scale, q, ldq, packed, colsum);
      break;
    }
    default: return -2;
  }
#undef SBQ_PACK2
#undef SBQ_PACK
  return check_launch();
}

int launch_parts_fill(const PartsFill& f, uint32_t begin4, int32_t* table, hipStream_t st) {
  const uint32_t n = f.end4[f.count - 1] - begin4;
  hipLaunchKernelGGL(parts_fill_kernel, dim3((n + 255) / 256), dim3(256), 0, st, f, begin4, table);
  return check_launch();
}

int launch_unpack(const uint8_t* packed, int64_t N, int64_t K, int8_t* q, int64_t ldq, hipStream_t st) {
  const int64_t Kc = (K + 63) / 64, nslots = (N + 15) / 16 * Kc * 64;
  hipLaunchKernelGGL(unpack_kernel, dim3((unsigned)((nslots + 255) / 256)), dim3(256), 0, st, packed, N, K, Kc, nslots,
                     q, ldq);
  return check_launch();
}

int minmax_nparts(int64_t M, int64_t K) {
  const int64_t total = M * K;
  int64_t p = (total + 2047) / 2048;  // >= 8 elements per thread at the smallest block
  if (p < 1) p = 1;
  if (p > kMinMaxPartials) p = kMinMaxPartials;
  return (int)p;
}

int launch_minmax_partials(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, float2* partials,
                           int nparts, hipStream_t st, uint32_t* zero, int nzero) {
  const int esz = xt == XT_F32 ? 4 : 2;
  const int vec = ((uintptr_t)x % 16 == 0) && ((ldx * esz) % 16 == 0);
  // smaller workgroups for small x (measured at K = 4096: M = 128 3.4 -> 2.8 us,
  // M = 512 3.6 -> 3.4 us; from M = 1024 the 1024-thread workgroups are fastest)
  const int64_t total = M * K;
  const int threads = total <= ((int64_t)1 << 19) ? 256 : (total <= ((int64_t)1 << 21) ? 512 : 1024);
  dim3 grid((unsigned)nparts), block(threads);
  if (vec && ldx == K && K % 8 == 0) {  // one flat array of 8-value chunks
    const int64_t nch = total / 8;
#define SBQ_MINMAX_DENSE(XT_)                                                                                    \
  hipLaunchKernelGGL((minmax_dense_kernel<XT_, 4>), grid, block, 0, st, x, nch, partials, zero, nzero);
    switch (xt) {
      case XT_F32: SBQ_MINMAX_DENSE(XT_F32) break;
      case XT_F16: SBQ_MINMAX_DENSE(XT_F16) break;
      case XT_BF16: SBQ_MINMAX_DENSE(XT_BF16) break;
      default: return -2;
    }
#undef SBQ_MINMAX_DENSE
    return check_launch();
  }
  switch (xt) {
    case XT_F32: hipLaunchKernelGGL(minmax_partial_kernel<XT_F32>, grid, block, 0, st, x, (int)M, (int)K, ldx, partials, vec, zero, nzero); break;
    case XT_F16: hipLaunchKernelGGL(minmax_partial_kernel<XT_F16>, grid, block, 0, st, x, (int)M, (int)K, ldx, partials, vec, zero, nzero); break;
    case XT_BF16: hipLaunchKernelGGL(minmax_partial_kernel<XT_BF16>, grid, block, 0, st, x, (int)M, (int)K, ldx, partials, vec, zero, nzero); break;
    default: return -2;
  }
  return check_launch();
}

int launch_qparams(const float2* partials, int nparts, float* scale_out, int32_t* zp_out, hipStream_t st) {
  hipLaunchKernelGGL(qparams_kernel, dim3(1), dim3(256), 0, st, partials, nparts, scale_out, zp_out);
  return check_launch();
}

int launch_rowsum_f16(const void* x, int64_t ldx, int64_t M, int64_t K, float* out, hipStream_t st, uint32_t* zero,
                      int nzero) {
  hipLaunchKernelGGL(rowsum_f16_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, st, (const _Float16*)x, ldx, (int)M,
                     (int)K, out, zero, nzero);
  return check_launch();
}

int launch_stage_act(const void* x, int xt, int64_t ldx, int64_t M, int64_t K, _Float16* xs, float* rowsum,
                     float* rscale, hipStream_t st, uint32_t* zero, int nzero) {
  const dim3 grid((unsigned)((M + 3) / 4)), block(256);
  if (xt == XT_F32)
    hipLaunchKernelGGL((stage_act_kernel<XT_F32, 8>), grid, block, 0, st, x, ldx, (int)M, (int)K, xs, rowsum, rscale,
                       zero, nzero);
  else if (xt == XT_BF16)
    hipLaunchKernelGGL((stage_act_kernel<XT_BF16, 8>), grid, block, 0, st, x, ldx, (int)M, (int)K, xs, rowsum, rscale,
                       zero, nzero);
  else
    return -2;
  return check_launch();
}

int launch_pad_rows(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, void* out, hipStream_t st, uint32_t* zero,
                    int nzero) {
  const int64_t cpr = (K + 63) / 64 * 8, nch = M * cpr;
  const dim3 grid((unsigned)((nch + 255) / 256)), block(256);
  switch (xt) {
    case XT_F32: hipLaunchKernelGGL((pad_rows_kernel<XT_F32, 1>), grid, block, 0, st, x, ldx, nch, (int)cpr, (int)K, (uint8_t*)out, zero, nzero); break;
    case XT_F16: hipLaunchKernelGGL((pad_rows_kernel<XT_F16, 1>), grid, block, 0, st, x, ldx, nch, (int)cpr, (int)K, (uint8_t*)out, zero, nzero); break;
    case XT_BF16: hipLaunchKernelGGL((pad_rows_kernel<XT_BF16, 1>), grid, block, 0, st, x, ldx, nch, (int)cpr, (int)K, (uint8_t*)out, zero, nzero); break;
    default: return -2;
  }
  return check_launch();
}

int launch_split_rows(const void* x, int64_t M, int64_t K, int64_t ldx, void* out, hipStream_t st, uint32_t* zero,
                      int nzero) {
  const int64_t cpr = (K + 63) / 64 * 8, nch = M * cpr;
  hipLaunchKernelGGL((pad_rows_kernel<XT_F32, 2>), dim3((unsigned)((nch + 255) / 256)), dim3(256), 0, st, x, ldx, nch,
                     (int)cpr, (int)K, (uint8_t*)out, zero, nzero);
  return check_launch();
}

int launch_act_quant_u8(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const float2* partials,
                        int nparts, uint8_t* xq, int64_t ldq, hipStream_t st) {
  const int64_t chunks = M * ((K + 7) / 8);
  const dim3 grid((unsigned)((chunks + 255) / 256)), block(256);
  const bool qvec = (uintptr_t)xq % 8 == 0 && ldq % 8 == 0;
  switch (xt) {
    case XT_F32: hipLaunchKernelGGL(act_quant_u8_kernel<XT_F32>, grid, block, 0, st, x, ldx, (int)M, (int)K, xvec, partials, nparts, xq, ldq, qvec); break;
    case XT_F16: hipLaunchKernelGGL(act_quant_u8_kernel<XT_F16>, grid, block, 0, st, x, ldx, (int)M, (int)K, xvec, partials, nparts, xq, ldq, qvec); break;
    case XT_BF16: hipLaunchKernelGGL(act_quant_u8_kernel<XT_BF16>, grid, block, 0, st, x, ldx, (int)M, (int)K, xvec, partials, nparts, xq, ldq, qvec); break;
    default: return -2;
  }
  return check_launch();
}

int launch_quantize_rows_sym(const void* x, int xt, int64_t ldx, bool xvec, int64_t M, int64_t K, int64_t Kp,
                             int8_t* xq, float* s_out, hipStream_t st, uint32_t* zero, int nzero) {
  const dim3 grid((unsigned)((M + 3) / 4)), block(256);
  const int vec = xvec ? 1 : 0;
  switch (xt) {
    case XT_F32: hipLaunchKernelGGL(quantize_rows_sym_kernel<XT_F32>, grid, block, 0, st, x, ldx, (int)M, (int)K, (int)Kp, vec, xq, s_out, zero, nzero); break;
    case XT_F16: hipLaunchKernelGGL(quantize_rows_sym_kernel<XT_F16>, grid, block, 0, st, x, ldx, (int)M, (int)K, (int)Kp, vec, xq, s_out, zero, nzero); break;
    case XT_BF16: hipLaunchKernelGGL(quantize_rows_sym_kernel<XT_BF16>, grid, block, 0, st, x, ldx, (int)M, (int)K, (int)Kp, vec, xq, s_out, zero, nzero); break;
    default: return -2;
  }
  return check_launch();
}

int launch_argmax_rows(const float* y, int64_t M, int64_t N, int64_t ldy, int64_t* out, hipStream_t st) {
  // rows that one workgroup takes several rounds of loads for (N = 8192, one
  // launch / three: 8.7 us / 6.0 in a graph, 8.7 / 8.5 eager, where the host's
  // launches count; N = 5000 8 / 6 and 7.6 / 8.5), until the rows alone fill the
  // chip (V = 151936, 256 rows: 51.3 us / 52.1; 64 rows 47.6 / 27.8)
  if (N >= 8192 && M <= 128) {
    unsigned long long* keys = (unsigned long long*)out;
    const int G = (int)min((N + 2047) / 2048, (int64_t)64), per = (int)((N + G - 1) / G);
    const dim3 rows((unsigned)((M + 255) / 256)), block(256);
    hipLaunchKernelGGL(argmax_clear_kernel, rows, block, 0, st, keys, M);
    hipLaunchKernelGGL(argmax_slice_kernel, dim3((unsigned)G, (unsigned)M), block, 0, st, y, (int)N, ldy, per, keys);
    hipLaunchKernelGGL(argmax_index_kernel, rows, block, 0, st, keys, M);
    return check_launch();
  }
  const int vec = ((uintptr_t)y % 16 == 0) && (ldy % 4 == 0);
  hipLaunchKernelGGL(argmax_rows_kernel, dim3((unsigned)M), dim3(1024), 0, st, y, (int)N, ldy, out, vec);
  return check_launch();
}

}  // namespace sbq
