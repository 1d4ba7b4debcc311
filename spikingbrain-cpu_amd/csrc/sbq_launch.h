// sbq_launch.h - internal host-side launchers shared between the kernel files
// and the C ABI (sbq_abi.hip).  Return 0 or a negative SBQ_ERR_* code.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sbq_common.h"

namespace sbq {

inline int check_launch() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : -5;
}

// One pass over weight rows (sbq_quant.hip pack_weight_kernel): wt a dtype
// (quantize_per_channel) or XT_S8 (rows as they are); scale is for a dtype
// only; q, packed, colsum: each may be null.
int launch_pack_weight(const void* w, int wt, int64_t N, int64_t K, int64_t ldw, float* scale, int8_t* q, int64_t ldq,
                       uint8_t* packed, int32_t* colsum, hipStream_t st);
// Table entries (see sbq_linear_w8_parts) of up to kPartsFill consecutive parts.
constexpr int kPartsFill = 16;
struct PartsFill {
  int count;
  uint32_t end4[kPartsFill];   // first 4-column group past each part
  uint32_t width[kPartsFill], word[kPartsFill];
};
int launch_parts_fill(const PartsFill& f, uint32_t begin4, int32_t* table, hipStream_t st);
int launch_unpack(const uint8_t* packed, int64_t N, int64_t K, int8_t* q, int64_t ldq, hipStream_t st);

int minmax_nparts(int64_t M, int64_t K);
// zero / nzero (optional): counters the pre-pass zeroes for the split-K GEMM
// launched after it on the same stream.
int launch_minmax_partials(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, float2* partials,
                           int nparts, hipStream_t st, uint32_t* zero = nullptr, int nzero = 0);
int launch_qparams(const float2* partials, int nparts, float* scale_out, int32_t* zp_out, hipStream_t st);
int launch_argmax_rows(const float* y, int64_t M, int64_t N, int64_t ldy, int64_t* out, hipStream_t st);
// The engine's non-greedy sampling step (sbq_sample.hip) over rows of fp32
// logits; ws: sample_workspace_bytes(M), 256-byte aligned.  Vocabularies up
// to kSampMaxVocab: a row's fixed-point mass (each token at most 2^40) then
// stays below 2^63.
constexpr int64_t kSampMaxVocab = (int64_t)1 << 23;
int64_t sample_workspace_bytes(int64_t M);
int launch_sample_rows(const float* x, int64_t M, int64_t V, int64_t ld, float T, int64_t top_k, float top_p,
                       const float* u, int64_t* tokens, void* ws, hipStream_t st);

// True when the streaming GEMV kernels take this M and K (otherwise the GEMM):
// up to 32 rows, and int8-dyn up to 16 of any x.
bool gemv_supports(int64_t M, int64_t K, bool w8a8, int xt);
// The general GEMV's configuration for an [M, K] input (sbq_gemv_config):
// info[0..8] = ok, row tiles of x, weight tiles per group, K tiles per wave,
// waves, activation mode, staging chunks per thread, LDS bytes, and whether a
// kernel instance exists for it.
int gemv_config_info(int64_t M, int64_t K, bool w8a8, int xt, int32_t* info);

// Decode fast path (sbq_gemv_fast.hip): M <= 16, K % 64 == 0, aligned x rows.
// pick_gemv_fast chooses a configuration id and the waves per workgroup;
// launch_gemv_fast_cfg returns -1 when that configuration cannot run the shape.
struct GemvArgs;
struct GemvSeg;
void pick_gemv_s8(int64_t M, int64_t K, int64_t N, int* id, int* ks);
bool gemv_quantize_first(int64_t M, int64_t K, int64_t N, int xt);
bool pick_gemv_fast(int64_t M, int64_t K, int64_t N, int xt, bool w8a8, bool xvec, int* id, int* ks,
                    bool token = false);
int launch_gemv_fast_cfg(int id, int ks, const GemvArgs& a, int xt, bool w8a8, hipStream_t st);
// Decode over several 16-row tiles of x (16 < M <= 64): weight-only on fp16 /
// bf16 x, or int8-dyn on pre-quantized s8 rows (xt XT_S8).  gemm_alt: the
// caller can run the tiled GEMM's mid-sized-M plan instead (then the path is
// taken on fewer shapes).
bool gemv_mt_applies(int64_t M, int64_t K, int64_t N, int xt, bool gemm_alt);
int launch_gemv_mt(const GemvArgs& a, int xt, hipStream_t st, bool gemm_alt);
int launch_gemv_w8_mt(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const uint8_t* packed,
                      const float* scale, const float* bias, int64_t N, void* y, int yt, int64_t ldy, hipStream_t st,
                      bool yvec, bool gemm_alt, const u32x2* parts = nullptr);
// Grouped launch: a.seg / a.nseg hold 2..kGemvMaxSeg linears (w8a8: int8-dyn
// with the activation min/max reduced in the kernel).
int launch_gemv_fast_grouped(int id, int ks, GemvArgs a, int xt, bool w8a8, hipStream_t st);
// n independent linears sharing M, K and dtypes in one launch (x / weight /
// scale / bias / colsum / y / strides / N / Nt per segment), weight-only or
// int8-dyn (w8a8); -1 when the fast path does not apply.
// With xq0 / qp0 (w8a8), inputs beyond the fused capacity are quantized first, in one launch, into
// xq0[i] and qp0[i].
int launch_gemv_w8_grouped(const GemvSeg* segs, int n, int xt, int64_t M, int64_t K, bool xvec, int yt, bool yvec,
                           hipStream_t st, bool w8a8 = false, int8_t* const* xq0 = nullptr,
                           float* const* qp0 = nullptr);

// Fused greedy token of the decode GEMV (fp32 y, M <= 16): the argmax state
// (kArgmaxStateBytes, zero before a launch, zero again after it) and the
// int64 token per row.  The launcher sets `fused` when the GEMV it ran also
// picked the tokens; otherwise the caller picks them from y.
struct GemvArgmaxOut {
  uint8_t* state;
  int64_t* idx;
  bool fused;
};

// parts (the linear launchers below): y stored as parts (part_base in
// sbq_index.h), one table entry per 4 columns; null: rows of stride ldy.
// Weight-only linear.  xvec: x and every row of x start 16-byte aligned (vector
// loads allowed).  yvec: y rows are 16-byte aligned and N % 4 == 0.
int launch_gemv_w8(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const uint8_t* packed,
                   const float* scale, const float* bias, int64_t N, void* y, int yt, int64_t ldy, hipStream_t st,
                   bool yvec, GemvArgmaxOut* am = nullptr, const u32x2* parts = nullptr);
// ws: device scratch (nullable, 256-byte aligned) of ws_bytes bytes, laid out
// by w8_ws_layout.  With enough of it the fp16 GEMM takes its per-row sums of x
// from a pre-pass, and fp32 / bf16 activations are staged as a scaled fp16
// plane for the same GEMM.
int launch_gemm_w8(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const uint8_t* packed,
                   const float* scale, const float* bias, int64_t N, void* y, int yt, int64_t ldy, void* ws,
                   int64_t ws_bytes, hipStream_t st, bool yvec, const u32x2* parts = nullptr);
// split: scratch after the workspace's layout (split_area_bytes of the plan;
// a shorter or null one runs the shape without splitting K).
// Direct-to-LDS GEMM plan: block configuration id and K splits (1: none);
// with splits, `tiles` output blocks of 64 x 64 and their partial tiles.
struct DlPlan {
  int id, splits;
  int64_t tiles, part_bytes;
};
DlPlan plan_gemm_dl(bool i8, int xt, int64_t M, int64_t Nt, int64_t Kc, bool rsp);
// Bytes of a plan's split-K scratch (0 without splits): tile counters, then
// the partial tiles; the GEMM launchers take it after their other scratch.
int64_t split_area_bytes(const DlPlan& p);

// W-only prefill scratch: [rowsum: M floats][rscale: M floats][fp16 plane: M x K for
// fp32 and bf16 x, none for fp16; ragged K: rows of whole tiles, two bf16
// planes for fp32], each part 256-byte aligned.
struct W8Ws {
  int64_t rowsum, rscale, planes, bytes;
};
W8Ws w8_ws_layout(int64_t M, int64_t K, int xt);
// Per-token symmetric W8A8 (opt-in int8-dyn granularity): xq scratch M x Kp
// bytes (Kp = ceil(K/64)*64), s_t scratch M floats.
int launch_gemm_w8a8_token(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec,
                           const uint8_t* packed, const float* scale, const float* bias, int64_t N, void* y, int yt,
                           int64_t ldy, int32_t* acc_out, int8_t* xq, float* s_t, hipStream_t st, bool yvec,
                           uint8_t* split, int64_t split_bytes);
// uint8 xq [M][ldq] of fbgemm's per-tensor activation quantization from the
// min/max partials (sbq_act_quant_per_tensor).
int launch_act_quant_u8(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const float2* partials,
                        int nparts, uint8_t* xq, int64_t ldq, hipStream_t st);
int launch_quantize_rows_sym(const void* x, int xt, int64_t ldx, bool xvec, int64_t M, int64_t K, int64_t Kp,
                             int8_t* xq, float* s_out, hipStream_t st, uint32_t* zero = nullptr, int nzero = 0);
// Per-row sums in fp32 of fp16 x [M, K] (K % 8 == 0, 16-byte aligned rows).
int launch_rowsum_f16(const void* x, int64_t ldx, int64_t M, int64_t K, float* out, hipStream_t st,
                      uint32_t* zero = nullptr, int nzero = 0);
// x [M, K] of any row stride, alignment and K as rows of Kp = ceil(K/64)*64
// columns, padding 0: a copy in x's dtype, and (fp32) bf16 high and remainder
// planes, [M][2][Kp].
int launch_pad_rows(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, void* out, hipStream_t st,
                    uint32_t* zero = nullptr, int nzero = 0);
// Whether a ragged weight-only call (K % 64 != 0) that the general GEMV takes
// (M <= 32) gains from rows of whole tiles, a launch more, on the fast GEMV (M <=
// 16) or the tiled GEMM: as K grows, and on wide layers.  xvec: the rows are
// 16-byte aligned as they are, which the general GEMV reads with vector loads.
// The lines lie where both sides are equal over 6000 timings in HIP graphs (N =
// 16 ... 150000, K = 65 ... 9000; us, general -> padded): 2999 x 2500, fp32 13.0
// -> 8.3 at 4 rows, one row 7.2 -> 8.4; fp16, 8 rows 8.8 -> 6.7 at N = 2999, K =
// 2500, but rows of 20 x 631 4.2 -> 6.7 and 36683 x 160 at 11 rows 6.6 -> 12.0;
// 11999 x 4000, fp32 31.5 -> 16.4 at 4 rows, 16.5 -> 12.8 at one; 1000 x 9001,
// fp32 24.5 -> 9.8 at one row, 60.2 -> 24.6 at 16; 20 rows of 2692 x 313, fp32 5.7
// -> 9.0; aligned fp16 rows at 28 x 2431 x 2168 1.7 times slower padded, 32 x
// 12780 x 3000 0.6 of it.
inline bool pad_ragged_rows(int64_t M, int64_t N, int64_t K, int xt, bool xvec) {
  const int64_t nk = (N * K) >> 20;
  // K >= k0, or weights of n1 MiB at K >= k1, or of n2 MiB
  const auto past = [&](int64_t k0, int64_t k1, int64_t n1, int64_t n2) {
    return K >= k0 || (K >= k1 && nk >= n1) || nk >= n2;
  };
  if (xt == 0) {
    if (M == 1) return past(4096, 512, 16, 32);
    if (M == 2) return xvec ? past(8192, 512, 8, 64) : past(384, 384, 0, 10);
    return past(M > 8 && M <= 16 ? 4096 : 1024, 256, 8, xvec ? 64 : 10);
  }
  if (M == 1) return false;
  if (xvec) {
    if (M <= 4) return past(M == 2 ? K + 1 : 6144, 512, 20, 64);
    return M <= 16 ? past(4096, 512, 10, 64) : past(4096, 1024, 20, 64);
  }
  if (M == 2) return past(1536, 512, 8, 24);
  return M <= 16 ? past(768, 320, 4, 12) : past(128, 128, 0, 6);
}
int launch_split_rows(const void* x, int64_t M, int64_t K, int64_t ldx, void* out, hipStream_t st,
                      uint32_t* zero = nullptr, int nzero = 0);
// fp32 / bf16 x [M, K] -> a scaled fp16 plane, row sums and row scales.
int launch_stage_act(const void* x, int xt, int64_t ldx, int64_t M, int64_t K, _Float16* xs, float* rowsum,
                     float* rscale, hipStream_t st, uint32_t* zero = nullptr, int nzero = 0);

// W8A8 (fbgemm dynamic semantics).  The decode fast path quantizes a small x
// in the kernel; a larger one, or ragged or misaligned rows, is quantized
// before it into xq (s8 [M][Kc*64]) and (s_x, zp) in qpbuf; above 16 rows its
// min/max goes into `partials` (>= kMinMaxPartials float2).
int launch_gemv_w8a8(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const uint8_t* packed,
                     const float* scale, const int32_t* colsum, const float* bias, int64_t N, void* y, int yt,
                     int64_t ldy, int32_t* acc_out, float2* partials, int8_t* xq, float* qpbuf, hipStream_t st,
                     bool yvec, GemvArgmaxOut* am = nullptr, const u32x2* parts = nullptr);
// Small activations quantized per tensor in one launch, one workgroup per
// input (quantize_small_fits): up to 4 inputs [M, K] of one dtype.
constexpr int kQuantSmallChunks = 20;  // 16-byte chunks of fp32 x per thread (1024 threads)
struct QuantSmall {
  const void* x[4];
  int64_t ldx[4];
  int8_t* xq[4];    // s8 rows xq - 128 [M][Kp]
  float* qpbuf[4];  // (s_x, zp bits)
  int M, K, Kp;     // Kp: K rounded up to 64
  uint32_t* zero;   // counters to clear (nullable)
  int nzero;
};
bool quantize_small_fits(int64_t M, int64_t K, int64_t Kp, int64_t ldx, bool xvec);
int launch_quantize_small(const QuantSmall& a, int count, int xt, hipStream_t st);
// ... or in two (min/max partials, then the rows) when x is larger.
int launch_quantize_acts(const void* x, int xt, int64_t M, int64_t K, int64_t Kp, int64_t ldx, bool xvec,
                         float2* partials, int8_t* xq, float* qpbuf, hipStream_t st, uint32_t* zero = nullptr,
                         int nzero = 0);
// The GEMM quantizes x once into xq (s8 [M][Kc*64]) and writes (s_x, zp) to
// qpbuf[0..1] (zp as int bits) before the tiled pipeline reads them.
int launch_gemm_w8a8(const void* x, int xt, int64_t M, int64_t K, int64_t ldx, bool xvec, const uint8_t* packed,
                     const float* scale, const int32_t* colsum, const float* bias, int64_t N, void* y, int yt,
                     int64_t ldy, int32_t* acc_out, float2* partials, int8_t* xq, float* qpbuf, hipStream_t st,
                     bool yvec, uint8_t* split = nullptr, int64_t split_bytes = 0,
                     const u32x2* parts = nullptr);

}  // namespace sbq
