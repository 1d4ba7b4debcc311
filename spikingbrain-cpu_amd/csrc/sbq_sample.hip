// sbq_sample.hip - the engine's sampling step on the GPU: temperature,
// top-k, top-p and the draw over the lm_head logits
// (spikingbrain_cpu/engine.py:29-42, paths relative to the reference
// repository), so that a non-greedy decode step leaves the logits on the GPU.
//
// Per row of fp32 logits x [V] (engine.py:29-42):
//   z = x / T                                 (IEEE fp32 division)
//   top_k > 0: kth = the k-th largest z (k = min(top_k, V)); z < kth is masked
//   p = softmax(z) = exp(z - max) / sum       (fp32)
//   0 < top_p < 1: a token is kept when the probability mass of the tokens
//   above it is below top_p (the reference's sorted `cumsum - p < top_p`)
//   token = the first index i (vocabulary order) whose prefix mass of kept
//   tokens exceeds u * (kept mass), u in [0, 1) supplied by the caller (the
//   inverse of the distribution torch.multinomial draws from).
//
// No sort.  Both cuts (the k-th largest z, the top-p boundary) are found in
// two levels.  The row's tokens are counted (top-k) and their masses
// exp(z - max), in 2^-40 fixed point, added (top-p) in kSampBins bins of z,
// laid between samples of the row (SampTable); a token more than 28 below the
// maximum has mass 0, and all of those share the last bin.  Every sum is an
// exact integer, independent of the order the atomics land in; top_p is applied
// to the kept mass as top_p * sum, which is the normalized condition.  The bins
// of the two cuts (or, while the kept mass still depends on the k-th token, the
// few bins its bounds allow) hold the only undecided tokens: a few hundred of
// 151936.  They are listed per slice, and one workgroup per row finds the exact
// keys among them (order-preserving 32-bit keys of z, 256 ranges per step), adds
// up the slices and draws.  Four launches for any cut: maximum and samples,
// bins, lists, draw (three without a cut).
//
// What bounds it: the launches and the latency of each one's serial chain;
// the logits (608 KB at V = 151936) are read from L2 three times.  Measured
// in a HIP graph at V = 151936 on one box, against one launch per 8 key bits of
// each cut over the whole row (7 launches with top-p, 10 with top-k as well): one
// row of a language model's logits, top-p 35.0 -> 20.7 us, top-k 50 and top-p 51.2
// -> 24.4, no cut 14.1 -> 12.3; eight rows, both cuts 67.2 -> 31.9.  Per launch at one
// row: 3.2 (maximum), 4.6, 4.8, 6.0 us.  Bins of equal width over the row's range
// took 20.4, 24.0 and 30.1 us there, but 390 (both cuts 470) on a flat row with one
// far or masked token; between samples such rows take 26 and 27, and no row of 19
// kinds (masked, clustered, tied, sorted) more than the radix launches did (top-p
// 38 at most).  Over many rows the vector units bound the bins launch (eight rows:
// 7.4 us, equal bins 5.8): a token takes 62 instructions, 38 with equal bins.
// 512 bins: 256 and 1024 of equal width ran within 2% at one row; 1024 was 25%
// slower at 16 rows (more atomics per slice).
//
// No workgroup waits for another: what a launch needs from the one before it
// (maximum, bins) every workgroup derives for itself.  Rows are independent
// (grid.y).  Differences from
// the reference's sort-based form: the top-p rule walks the tokens in the
// order of z, where the sort walks the fp32 probabilities, so of two tokens
// whose probabilities round to the same fp32 value the larger z comes first
// (the sort leaves the order of equal values open); and a token's mass is
// exp(z - max) truncated to 2^-40.  Tokens whose z ties at the top-p boundary
// are kept as the sort keeps them: as many as its rule admits, the first ones
// in vocabulary order (the order a stable sort gives them).
#include <stdint.h>

#include "sbq_common.h"
#include "sbq_launch.h"

namespace sbq {

constexpr int kSampThreads = 1024;
constexpr int kSampWaves = kSampThreads / 64;
constexpr int kSampMaxBlocks = 64;   // workgroups (slices) per row: one wave's lanes hold a value of each
constexpr int kSampBins = 512;       // bins of z
constexpr int kSampCopies = 8;       // LDS copies of each bin (atomics of one wave spread over them)
constexpr int kSampUnroll = 4;       // tokens in flight per thread
constexpr int kSampList = 1024;      // undecided tokens listed per slice (a slice with more is read again)
constexpr int kSampFew = 32;         // a slice with more undecided tokens looks whether they share one key
constexpr uint32_t kSampTied = 1u << 31;  // ... and they do: the list's first place holds it
constexpr float kSampRange = 28.0f;  // exp(-28) < 2^-40: a mass of 0 from here down

// Per-row scratch, from the row's first byte (each part 256-byte aligned).
struct SampRow {
  static constexpr int64_t kHead = 0;                      // SampHead
  static constexpr int64_t kMax = 256;                     // float [G]
  static constexpr int64_t kMin = kMax + 256;              // float [G]
  static constexpr int64_t kNan = kMin + 256;              // int [G]
  static constexpr int64_t kSplit = kNan + 256;            // float [64]: samples of z, largest first
  static constexpr int64_t kSum = kSplit + 256;            // uint64 [G]: mass above every undecided bin
  static constexpr int64_t kNum = kSum + 512;              // uint32 [G]: undecided tokens of the slice (| kSampTied)
  static constexpr int64_t kMass = kNum + 256;             // uint64 [kSampBins]
  static constexpr int64_t kCount = kMass + kSampBins * 8; // uint32 [kSampBins]
  static constexpr int64_t kList = kCount + kSampBins * 4; // uint32 [G][kSampList]: keys of the undecided tokens
  static constexpr int64_t kBytes = kList + kSampMaxBlocks * kSampList * 4;
};
static_assert(kSampMaxBlocks * 8 <= 512 && kSampMaxBlocks * 4 <= 256 && kSampMaxBlocks <= 64,
              "per-slice arrays fit their slots and one wave");
static_assert(kSampMaxBlocks == 64, "one lane per slice, its number in seven bits");
static_assert(kSampMaxBlocks % kSampWaves == 0, "the draw's waves own whole sets of slices");

// The undecided bins of a row, recorded by the list launch for the draw.
struct SampHead {
  int valid;      // 0: a NaN or an infinite max (the reference raises)
  float m, low;   // max z; the lowest z that the bins resolve
  int kbin;       // the bin of the k-th largest z (-1: top-k masks nothing of mass)
  int krest;      // its rank within that bin, from the top
  int lo, hi;     // the top-p boundary lies in bins lo .. hi (lo > hi: no top-p)
  int pad;
  uint64_t kabove;  // mass of the bins above kbin
  uint64_t labove;  // mass of the bins above lo
  uint64_t total;   // mass of the row
};

struct SampArgs {
  const float* x;
  int64_t ld;
  int V, G, per;
  float T;
  int k;                 // min(top_k, V), or 0
  double top_p;          // 0 without top-p
  uint8_t* ws;
  const float* u;        // [M] uniforms in [0, 1)
  int64_t* tokens;       // [M]
};

// Order-preserving key: a < b as floats <=> key(a) < key(b); -0 as +0.
__device__ __forceinline__ uint32_t samp_key(float z) {
  const uint32_t b = __float_as_uint(z == 0.0f ? 0.0f : z);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// z of a key (the inverse of samp_key; +0 for the key of zeros)
__device__ __forceinline__ float samp_unkey(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ float samp_z(const SampArgs& a, const float* row, int i) { return row[i] / a.T; }

// fixed-point mass exp(z - m) * 2^40, truncated: exp(z - m) <= 1 in units of
// 2^-16, then the rest of them in units of 2^-24 (every step but the two
// truncations exact)
__device__ __forceinline__ uint64_t samp_efix(float z, float m) {
  const float f = expf(z - m) * 65536.0f;
  const uint32_t hi = (uint32_t)f, lo = (uint32_t)((f - (float)hi) * 16777216.0f);
  return (uint64_t)hi << 24 | lo;
}

// The bins of a row: 64 sampled z, sorted, give 14 splits of the values into
// intervals of a few 64ths of the tokens each, whatever their distribution
// (equal steps of max - z put most of a flat row beside one far token into one
// bin, and one workgroup then read the row again per pass: 390 us at V =
// 151936).  Interval i lies below split i - 1 (the maximum); its first bin holds
// the tokens equal to that (ties), the rest are equal steps down to split i
// (in the last interval to `low`, the lowest z that can have mass): kSampTop of
// them in the first interval, where sampled decoding cuts, kSampSteps in the
// others.  A last split, the largest z below max - kSampRange, leaves the last
// bin to tokens without mass, and splits below it count as it.  Comparisons,
// rounding and ceil are monotone, so a larger z never has a larger bin, and
// equal z share one.
constexpr int kSampSplits = 14;
constexpr int kSampTop = 200, kSampSteps = 21;
static_assert(kSampSplits == 14, "the last split is the 15th, of a search in four steps");
static_assert(kSampTop + 1 + (kSampSteps + 1) * kSampSplits < kSampBins, "the intervals' bins and the last one");
// Split t of the row is sample samp_split(t), finer towards the top.
__device__ __forceinline__ int samp_split(int t) {
  return t < 2 ? t : (t < 4 ? 4 * t - 5 : (27 * t - 46) / 5);  // 0, 1, 3, 7, 12 ... 61
}
struct SampTable {
  float s[16];     // the splits, largest first
  f32x4 from[16];  // per interval: its top, steps per unit of z, steps, (int bits) first bin
};
// (Splits compared two levels deep or all at once, from scalar registers, and four
// tokens looked up together were slower: 0.3 to 1.5 us of the bins launch at
// eight rows.)
struct SampLook {
  const SampTable* tb;
  __device__ __forceinline__ int bin(float z) const {
    int i = 0;  // splits at or above z
#pragma unroll
    for (int step = 8; step > 0; step >>= 1) i += tb->s[i + step - 1] >= z ? step : 0;
    const f32x4 f = tb->from[i];
    return (int)__float_as_uint(f[3]) + (int)__builtin_ceilf(fminf((f[0] - z) * f[1], f[2]));
  }
};

// This lane's split (lane t: split t), for samp_table: one load, to be issued
// ahead of what the caller still has to find out.
__device__ __forceinline__ float samp_lane_split(const uint8_t* w) {
  return ((const float*)(w + SampRow::kSplit))[samp_split(min((int)(threadIdx.x & 63), kSampSplits - 1))];
}
// v of the lane before, within each 16 lanes
__device__ __forceinline__ float samp_lane_before(float v) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x111, 0xf, 0xf, false));
}

// (one wave: a lane per interval)
__device__ __forceinline__ void samp_table(float lane_split, float m, float low, SampTable* tb) {
  const int t = threadIdx.x & 63;
  const float bound = samp_unkey(samp_key(m - kSampRange) - 1u);
  const float split = t < kSampSplits ? fmaxf(lane_split, bound) : bound, before = samp_lane_before(split);
  if (t < 16) {
    const float top = t == 0 ? m : before, n = t == 0 ? (float)kSampTop : (t <= kSampSplits ? (float)kSampSteps : 0.0f);
    const float width = top - fmaxf(split, low);
    const int base = t == 0 ? 0 : (t <= kSampSplits ? kSampTop + 1 + (kSampSteps + 1) * (t - 1) : kSampBins - 1);
    tb->s[t] = split;
    tb->from[t] = (f32x4){top, width > 0.0f ? n / fmaxf(width, 1e-30f) : 0.0f, n, __uint_as_float((uint32_t)base)};
  }
}

// Tokens whose bin is sure to lie after `last`, without the lookup: those of a
// later interval, or past its step in bin()'s own arithmetic (the list launch,
// which needs only the others: 5.4 -> 4.8 us at one row, 7.9 -> 6.2 at eight).
struct SampAfter {
  float top, steps, end, step;
  __device__ __forceinline__ SampAfter(const SampTable* tb, int last)
      : top(0.0f), steps(0.0f), end(-INFINITY), step(INFINITY) {
    if (last < 0 || last >= kSampBins - 1) return;  // uniform: no bins, or none after it
    const int q = last - (kSampTop + 1), i = q < 0 ? 0 : 1 + q / (kSampSteps + 1);
    const int j = q < 0 ? last : q % (kSampSteps + 1);  // 0: the ties
    top = tb->from[i][0];
    steps = tb->from[i][1];
    end = tb->s[i];
    if (j < (i == 0 ? kSampTop : kSampSteps)) step = (float)j;
  }
  __device__ __forceinline__ bool operator()(float z) const { return z <= end || (top - z) * steps > step; }
};

// The top-p bound on the mass above a token: mass_above < top_p * S (S: the
// mass top-k keeps) <=> mass_above < thr, for integer masses.
__device__ __forceinline__ uint64_t samp_thr(double top_p, uint64_t S) { return (uint64_t)ceil(top_p * (double)S); }

__device__ __forceinline__ uint8_t* samp_row_ws(const SampArgs& a) { return a.ws + (int64_t)blockIdx.y * SampRow::kBytes; }

// The tokens [i0, i1) of the row as `n` consecutive threads, of which this is
// number `t`, take them: kSampUnroll loads in flight, indexes clamped to the
// range, surplus ones skipped.  The first round is loaded on construction
// (ahead of what the caller still has to find out: an L2 latency less per
// launch).
struct SampTokens {
  const float* row;
  int i0, i1, t, n;
  float x[kSampUnroll];

  __device__ __forceinline__ SampTokens(const float* row_, int i0_, int i1_, int t_, int n_)
      : row(row_), i0(i0_), i1(i1_), t(t_), n(n_) {
    load(i0 + t);
  }
  __device__ __forceinline__ void load(int b) {
#pragma unroll
    for (int u = 0; u < kSampUnroll; ++u) x[u] = row[max(min(b + u * n, i1 - 1), 0)];
  }
  // f(z[kSampUnroll], b) for each round: the tokens b + u n, those past the
  // range repeating its last one
  template <typename F>
  __device__ __forceinline__ void rounds(float T, F f) {
    for (int b = i0 + t; b < i1; b += kSampUnroll * n) {
      if (b != i0 + t) load(b);
      float z[kSampUnroll];
#pragma unroll
      for (int u = 0; u < kSampUnroll; ++u) z[u] = x[u] / T;
      f(z, b);
    }
  }
  // f(i, z) for each token
  template <typename F>
  __device__ __forceinline__ void each(float T, F f) {
    for (int b = i0 + t; b < i1; b += kSampUnroll * n) {
      if (b != i0 + t) load(b);
#pragma unroll
      for (int u = 0; u < kSampUnroll; ++u)
        if (b + u * n < i1) f(b + u * n, x[u] / T);
    }
  }
};

// v of the lane that the DPP control names, 0 where it names none
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t samp_dpp0(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ uint64_t samp_dpp0(uint64_t v) {
  return (uint64_t)samp_dpp0<CTRL, ROWS>((uint32_t)v) | (uint64_t)samp_dpp0<CTRL, ROWS>((uint32_t)(v >> 32)) << 32;
}

// Inclusive prefix sum over the lanes of one wave: within the rows of 16
// lanes, then across them (lane moves, no LDS round trips).
template <typename T>
__device__ __forceinline__ T wave_prefix(T v) {
  v += samp_dpp0<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v += samp_dpp0<0x112, 0xf>(v);
  v += samp_dpp0<0x114, 0xf>(v);
  v += samp_dpp0<0x118, 0xf>(v);
  v += samp_dpp0<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += samp_dpp0<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
// The last lane's value.
__device__ __forceinline__ uint32_t wave_last(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 63); }
__device__ __forceinline__ uint64_t wave_last(uint64_t v) {
  return (uint64_t)wave_last((uint32_t)v) | (uint64_t)wave_last((uint32_t)(v >> 32)) << 32;
}
template <typename T>
__device__ __forceinline__ T wave_total(T v) { return wave_last(wave_prefix(v)); }

// Block sum, every thread the result.  red: kSampWaves words, reused after
// the caller's next barrier.
__device__ __forceinline__ uint64_t samp_block_sum_u64(uint64_t v, uint64_t* red) {
  const int lane = threadIdx.x & 63;
  v = wave_total(v);
  if (lane == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return wave_total(lane < kSampWaves ? red[lane] : (uint64_t)0);
}

// A lowest z beside its tokens' largest one `mx`, once the largest is `top`:
// dropped when those are without mass beside it (masked slices).
__device__ __forceinline__ float samp_near(float mx, float top, float mn) {
  return mx >= top - kSampRange ? mn : INFINITY;
}

// The row's maximum, the lowest z the bins resolve, and validity from the
// first launch's per-slice values (identical in every wave and workgroup).
struct SampScale {
  float m, low;
  bool valid;
};
__device__ __forceinline__ SampScale samp_scale(const SampArgs& a, const uint8_t* w) {
  const int lane = threadIdx.x & 63, g = min(lane, a.G - 1);
  const float mxl = ((const float*)(w + SampRow::kMax))[g], mnl = ((const float*)(w + SampRow::kMin))[g];
  const int nl = ((const int*)(w + SampRow::kNan))[g];
  SampScale s;
  s.m = wave_max(mxl);
  s.low = fmaxf(wave_min(samp_near(mxl, s.m, mnl)), s.m - kSampRange);
  s.valid = __ballot(nl != 0) == 0 && s.m < INFINITY && s.m > -INFINITY;
  return s;
}

// The same, and with TABLE the bins' table, by one wave for its workgroup (all 16
// waves reading the row's three or four lines: the bins launch 0.4 us longer at
// eight rows, 0.3 at one).
template <bool TABLE>
__device__ __forceinline__ void samp_scale_table(const SampArgs& a, const uint8_t* w, SampScale* out, SampTable* tb) {
  const float split = TABLE ? samp_lane_split(w) : 0.0f;
  const SampScale sc = samp_scale(a, w);
  if constexpr (TABLE) samp_table(split, sc.m, sc.low, tb);
  if ((threadIdx.x & 63) == 0) *out = sc;
}

// The row's 64 samples, one in each 64th of the row (the place within it by the
// golden ratio), sorted: each of four waves ranks the lanes' samples against
// its sixteen, one adds up the ranks.  (On cold logits the launch takes 3.7 us
// so, 4.0 with four ranks in each of 16 waves, which all load the 64
// scattered samples, and 4.2 with two waves.)
constexpr int kSampRankWaves = 4, kSampRanks = 64 / kSampRankWaves;
__device__ __forceinline__ float samp_sample(const SampArgs& a) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t V = (uint64_t)a.V, turn = (uint64_t)(lane * 2654435769u) * V >> 32;
  return samp_z(a, a.x + (int64_t)blockIdx.y * a.ld, (int)((lane * V + turn) >> 6));
}
__device__ __forceinline__ int samp_rank(float z) {
  const int lane = threadIdx.x & 63, j0 = (threadIdx.x >> 6) * kSampRanks;
  int rank = 0;
#pragma unroll
  for (int j = j0; j < j0 + kSampRanks; ++j) {
    const float o = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(z), j));
    rank += o > z || (o == z && j < lane);
  }
  return rank;
}

// First launch: max z, min z of the tokens near it, and the NaN count per
// slice; workgroup 0 clears the row's bins and sorts its samples.
__global__ __launch_bounds__(kSampThreads) void samp_max_kernel(SampArgs a) {
  __shared__ float smx[kSampWaves], smn[kSampWaves];
  __shared__ int snan[kSampWaves], ranks[kSampRankWaves][64];
  uint8_t* w = samp_row_ws(a);
  const bool sort = blockIdx.x == 0 && threadIdx.x < kSampRankWaves * 64 && (a.k > 0 || a.top_p > 0.0);
  const int i0 = blockIdx.x * a.per, i1 = min(i0 + a.per, a.V);
  SampTokens tok(a.x + (int64_t)blockIdx.y * a.ld, i0, i1, threadIdx.x, kSampThreads);
  if (blockIdx.x == 0 && threadIdx.x < kSampBins) {
    ((uint64_t*)(w + SampRow::kMass))[threadIdx.x] = 0;
    ((uint32_t*)(w + SampRow::kCount))[threadIdx.x] = 0;
  }
  const int lane = threadIdx.x & 63;
  const float sample = sort ? samp_sample(a) : 0.0f;
  float mx = -INFINITY, mn = INFINITY;
  bool nan = false;
  tok.rounds(a.T, [&](const float (&z)[kSampUnroll], int) {
    float top = mx;
#pragma unroll
    for (int u = 0; u < kSampUnroll; ++u) {
      nan |= z[u] != z[u];
      top = fmaxf(top, z[u]);
    }
    mn = samp_near(mx, top, mn);
#pragma unroll
    for (int u = 0; u < kSampUnroll; ++u) mn = fminf(mn, samp_near(z[u], top, z[u]));
    mx = top;
  });
  float top = wave_max(mx);
  mn = wave_min(samp_near(mx, top, mn));
  mx = top;
  const int any = __ballot(nan) != 0;
  if (sort) ranks[threadIdx.x >> 6][lane] = samp_rank(sample);
  if (lane == 0) {
    smx[threadIdx.x >> 6] = mx;
    smn[threadIdx.x >> 6] = mn;
    snan[threadIdx.x >> 6] = any;
  }
  __syncthreads();
  if (threadIdx.x < 64) {  // wave 0: a lane per wave's values
    const int wv = min(lane, kSampWaves - 1);
    top = wave_max(smx[wv]);
    mn = wave_min(samp_near(smx[wv], top, smn[wv]));
    const int bad = __ballot(snan[wv] != 0) != 0;
    if (lane == 0) {
      ((float*)(w + SampRow::kMax))[blockIdx.x] = top;
      ((float*)(w + SampRow::kMin))[blockIdx.x] = mn;
      ((int*)(w + SampRow::kNan))[blockIdx.x] = bad;
    }
  } else if (sort && threadIdx.x < 128) {
    int rank = 0;
#pragma unroll
    for (int i = 0; i < kSampRankWaves; ++i) rank += ranks[i][lane];
    ((float*)(w + SampRow::kSplit))[min(rank, 63)] = sample;  // (a NaN: the row is invalid)
  }
}

// Second launch (with a cut): token counts (K: top-k) and masses (P: top-p)
// per bin, in LDS, then added into the row's bins.
template <bool K, bool P>
__global__ __launch_bounds__(kSampThreads) void samp_bins_kernel(SampArgs a) {
  __shared__ uint64_t H[P ? kSampBins * kSampCopies : 1];
  __shared__ uint32_t C[K ? kSampBins * kSampCopies : 1];
  __shared__ SampTable tb;
  __shared__ SampScale sc;
  uint8_t* w = samp_row_ws(a);
  const int i0 = blockIdx.x * a.per, i1 = min(i0 + a.per, a.V);
  SampTokens tok(a.x + (int64_t)blockIdx.y * a.ld, i0, i1, threadIdx.x, kSampThreads);
  if (threadIdx.x < 64) samp_scale_table<true>(a, w, &sc, &tb);
  for (int i = threadIdx.x; i < kSampBins * kSampCopies; i += kSampThreads) {
    if constexpr (P) H[i] = 0;
    if constexpr (K) C[i] = 0;
  }
  __syncthreads();
  if (!sc.valid) return;
  const float m = sc.m;
  const SampLook look{&tb};
  const int copy = threadIdx.x & (kSampCopies - 1);
  tok.each(a.T, [&](int, float z) {
    const int at = look.bin(z) * kSampCopies + copy;
    if constexpr (P) {
      const uint64_t f = samp_efix(z, m);
      if (f) atomicAdd((unsigned long long*)&H[at], (unsigned long long)f);
    }
    if constexpr (K) atomicAdd(&C[at], 1u);
  });
  __syncthreads();
  for (int b = threadIdx.x; b < kSampBins; b += kSampThreads) {
    if constexpr (P) {
      uint64_t s = 0;
#pragma unroll
      for (int c = 0; c < kSampCopies; ++c) s += H[b * kSampCopies + c];
      if (s) __hip_atomic_fetch_add((unsigned long long*)(w + SampRow::kMass) + b, (unsigned long long)s,
                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if constexpr (K) {
      uint32_t s = 0;
#pragma unroll
      for (int c = 0; c < kSampCopies; ++c) s += C[b * kSampCopies + c];
      if (s) __hip_atomic_fetch_add((uint32_t*)(w + SampRow::kCount) + b, s, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// The undecided bins of the row from its filled bins (identical in every
// workgroup).  Thread b < kSampBins holds bin b.
template <bool K, bool P>
__device__ void samp_cuts(const SampArgs& a, uint64_t f, uint32_t c, SampHead* h, uint64_t* red) {
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  constexpr int W = kSampBins / 64;
  uint64_t fi = P ? wave_prefix(f) : 0;
  uint32_t ci = K ? wave_prefix(c) : 0;
  if (lane == 63 && wv < W) {
    red[wv] = fi;
    red[W + wv] = ci;
  }
  __syncthreads();  // (the caller's *h as well)
  uint64_t total = 0;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    if (i < wv) {
      fi += red[i];
      ci += (uint32_t)red[W + i];
    }
    total += red[i];
  }
  const uint64_t fa = fi - f;  // mass of the bins above this one
  if constexpr (K) {
    // the bin of the k-th largest z; among the tokens without mass it cuts nothing
    const uint32_t ca = ci - c, k = (uint32_t)a.k;
    if (t < kSampBins && ca < k && k <= ci && t < kSampBins - 1) {
      h->kbin = t;
      h->krest = (int)(k - ca);
      h->kabove = fa;
      red[2 * W] = fi;
    }
    __syncthreads();
  }
  if constexpr (P) {
    const int kbin = K ? h->kbin : -1, last = kbin >= 0 ? kbin : kSampBins - 1;
    // the mass top-k keeps: known without it, else from that of the bins
    // above the k-th token's to that with its whole bin
    const uint64_t s0 = kbin >= 0 ? h->kabove : total, s1 = kbin >= 0 ? red[2 * W] : total;
    const uint64_t t0 = max(samp_thr(a.top_p, s0), (uint64_t)1), t1 = max(samp_thr(a.top_p, s1), (uint64_t)1);
    // the boundary's bin for a bound thr: the last one (down to the k-th
    // token's) whose mass above stays below thr
    if (t <= last) {
      if (fa < t0 && (t == last || fi >= t0)) {
        h->lo = t;
        h->labove = fa;
      }
      if (fa < t1 && (t == last || fi >= t1)) h->hi = t;
    }
    if (t == 0) h->total = total;
    __syncthreads();
  }
}

// Third launch: per slice, the mass of the tokens above every undecided bin
// and the list of the tokens in them.  A slice of many that all share one key
// (ties) records that key once, in the list's first place, and kSampTied in the
// count.
template <bool K, bool P>
__global__ __launch_bounds__(kSampThreads) void samp_list_kernel(SampArgs a) {
  __shared__ SampHead h;
  __shared__ uint64_t red[2 * (kSampBins / 64) + 1], sum[kSampWaves];
  __shared__ uint32_t num, kmin, kmax;
  __shared__ SampTable tb;
  __shared__ SampScale sc;
  uint8_t* w = samp_row_ws(a);
  const int i0 = blockIdx.x * a.per, i1 = min(i0 + a.per, a.V);
  SampTokens tok(a.x + (int64_t)blockIdx.y * a.ld, i0, i1, threadIdx.x, kSampThreads);
  uint64_t f = 0;
  uint32_t c = 0;
  if (threadIdx.x < kSampBins) {
    if constexpr (P) f = ((const uint64_t*)(w + SampRow::kMass))[threadIdx.x];
    if constexpr (K) c = ((const uint32_t*)(w + SampRow::kCount))[threadIdx.x];
  }
  if (threadIdx.x < 64) samp_scale_table<K || P>(a, w, &sc, &tb);
  if (threadIdx.x == 0) {
    num = 0;
    kmin = ~0u;
    kmax = 0;
    h = SampHead{1, sc.m, sc.low, -1, 0, 1, 0, 0, 0, 0, 0};  // (sc: this lane's own store)
  }
  if constexpr (K || P)
    samp_cuts<K, P>(a, f, c, &h, red);
  else
    __syncthreads();
  if (!sc.valid) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ((SampHead*)(w + SampRow::kHead))->valid = 0;
    return;
  }
  const float m = sc.m;
  const SampLook look{&tb};
  const int lo = h.lo, hi = h.hi, kbin = h.kbin;
  const SampAfter after(&tb, K || P ? max(lo <= hi ? hi : -1, kbin) : -1);  // most of a usual row
  // tokens above the first undecided bin are kept, whatever the keys say
  const int first = lo <= hi ? lo : (kbin >= 0 ? kbin : kSampBins);
  uint32_t* list = (uint32_t*)(w + SampRow::kList) + blockIdx.x * kSampList;
  uint64_t part = 0;
  uint32_t k0 = ~0u, k1 = 0;
  tok.each(a.T, [&](int, float z) {
    if ((K || P) && after(z)) return;
    const int b = K || P ? look.bin(z) : 0;
    if (b < first) {
      part += samp_efix(z, m);
    } else if (b <= hi || b == kbin) {
      const uint32_t at = atomicAdd(&num, 1u), k = samp_key(z);
      if (at < (uint32_t)kSampList) list[at] = k;
      k0 = min(k0, k);
      k1 = max(k1, k);
    }
  });
  part = samp_block_sum_u64(part, sum);
  const bool many = num > (uint32_t)kSampFew;  // uniform
  if (many) {
    if (k0 <= k1) {
      atomicMin(&kmin, k0);
      atomicMax(&kmax, k1);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const bool tied = many && kmin == kmax;
    if (tied) list[0] = kmin;
    ((uint64_t*)(w + SampRow::kSum))[blockIdx.x] = part;
    ((uint32_t*)(w + SampRow::kNum))[blockIdx.x] = num | (tied ? kSampTied : 0u);
    if (blockIdx.x == 0) *(SampHead*)(w + SampRow::kHead) = h;
  }
}

// The undecided tokens of the row in the draw: gathered through LDS, up to
// kFlat per thread in registers (the usual case: a few hundred, one per
// thread).  When there are more, on each use wave wv goes over the lists of
// the slices wv, wv + 16, ... (their one key if all tied), and all waves
// together over the logits of the slices with more than a list.
struct SampUndecided {
  static constexpr int S = kSampMaxBlocks / kSampWaves;
  static constexpr int kFlat = 4;
  bool flat;
  int sets;  // flat: ceil(tokens / kSampThreads)
  uint32_t key[kFlat], n[kFlat];  // n tokens of that key
  uint64_t mass[kFlat];
  int slice[kFlat];  // -1: none
  uint32_t num[S];   // tokens of this wave's slices, not flat
  uint64_t longer;   // slices to read again

  // lk, ls, lc: kFlat * kSampThreads words / bytes and kSampMaxBlocks words of LDS
  __device__ __forceinline__ void load(const SampArgs& a, const uint8_t* w, float m, uint32_t* lk, uint8_t* ls,
                                       uint32_t* lc) {
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const uint32_t* lists = (const uint32_t*)(w + SampRow::kList);
    uint32_t nl = ((const uint32_t*)(w + SampRow::kNum))[min(lane, a.G - 1)], k[S];
#pragma unroll
    for (int s = 0; s < S; ++s) k[s] = lists[min(wv + s * kSampWaves, a.G - 1) * kSampList + lane];
    if (lane >= a.G) nl = 0;
    longer = __ballot(nl > (uint32_t)kSampList && !(nl & kSampTied));
    const uint32_t el = nl & kSampTied ? 1u : (longer ? 0u : nl);  // entries
    const uint32_t incl = wave_prefix(el);
    const int total = (int)wave_last(incl);
    flat = !longer && total <= kFlat * kSampThreads;
    if (wv == 0) lc[lane] = nl & ~kSampTied;
    sets = (total + kSampThreads - 1) / kSampThreads;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int g = wv + s * kSampWaves;
      num[s] = (uint32_t)__builtin_amdgcn_readlane((int)nl, g);
      if (flat) {
        const int o = __builtin_amdgcn_readlane((int)(incl - el), g), e = __builtin_amdgcn_readlane((int)el, g);
        const uint8_t tied = num[s] & kSampTied ? 0x80 : 0;
#pragma unroll 4
        for (int j = lane; j < e; j += 64) {
          lk[o + j] = j < 64 ? k[s] : lists[g * kSampList + j];
          ls[o + j] = (uint8_t)g | tied;
        }
      }
    }
    __syncthreads();
    if (flat) {
#pragma unroll
      for (int i = 0; i < kFlat; ++i) {
        slice[i] = -1;
        if (i < sets) {
          const int at = t + i * kSampThreads;
          key[i] = lk[at];
          if (at < total) {
            const int g = ls[at];
            slice[i] = g & 0x7f;
            n[i] = g & 0x80 ? lc[slice[i]] : 1u;
          }
          mass[i] = samp_efix(samp_unkey(key[i]), m);  // (past the end: unused)
        }
      }
    }
  }

  // f(key, mass, n, slice) for the keys in [lo, hi], n tokens of that mass each
  template <typename F>
  __device__ __forceinline__ void each(const SampArgs& a, const uint8_t* w, const float* row, const SampHead& h,
                                       const SampLook& look, uint32_t lo, uint32_t hi, F f) const {
    if (flat) {
#pragma unroll
      for (int i = 0; i < kFlat; ++i)
        if (i < sets && slice[i] >= 0 && key[i] >= lo && key[i] <= hi) f(key[i], mass[i], n[i], slice[i]);
      return;
    }
    const int lane = threadIdx.x & 63;
    const auto one = [&](uint32_t k, uint32_t n, int g) {
      if (k >= lo && k <= hi) f(k, samp_efix(samp_unkey(k), h.m), n, g);
    };
#pragma unroll 1
    for (int s = 0; s < S; ++s) {
      const int g = (threadIdx.x >> 6) + s * kSampWaves;
      const uint32_t n = s == 0 ? num[0] : (s == 1 ? num[1] : (s == 2 ? num[2] : num[3]));
      const uint32_t* list = (const uint32_t*)(w + SampRow::kList) + g * kSampList;
      if (n <= (uint32_t)kSampList) {
        for (int j = lane; j < (int)n; j += 64) one(list[j], 1u, g);
      } else if (n & kSampTied) {
        if (lane == 0) one(list[0], n & ~kSampTied, g);
      }
    }
#pragma unroll 1
    for (uint64_t rest = longer; rest; rest &= rest - 1) {
      const int g = __ffsll((long long)rest) - 1, i1 = min((g + 1) * a.per, a.V);
#pragma unroll 1
      for (int i = g * a.per + (int)threadIdx.x; i < i1; i += kSampThreads) {
        const float z = samp_z(a, row, i);
        const int b = look.bin(z);
        if ((b >= h.lo && b <= h.hi) || b == h.kbin) one(samp_key(z), 1u, g);
      }
    }
  }
};
static_assert(SampUndecided::S == 4, "each() names the four counts");

// The cut among the undecided keys [lo, hi] (the lowest and highest present),
// by 256 equal ranges of keys per step until one key is left.  Counts (MASS
// false): the key of rank `rest` from the top.  Masses: the lowest key whose
// mass above it, `rest` on entry for `hi`, stays below thr; `rest` then is
// that mass.  H: kCutWords of LDS, range-major per copy.
constexpr int kCutCopies = 4;
constexpr int kCutStride = 256 + 2;  // copies of one range lie in different banks
constexpr int kCutWords = kCutCopies * kCutStride;
template <bool MASS>
__device__ __forceinline__ uint32_t samp_descend(const SampArgs& a, const uint8_t* w, const float* row, const SampHead& h,
                                 const SampUndecided& und, const SampLook& look, uint32_t lo, uint32_t hi, uint64_t& rest, uint64_t thr,
                                 uint64_t* H, uint64_t* bc) {
  const int t = threadIdx.x, lane = t & 63;
  uint64_t* const Hc = H + (lane & (kCutCopies - 1)) * kCutStride;
  while (lo < hi) {
    const int shift = max(0, 24 - (int)__clz((int)(hi - lo)));
    for (int i = t; i < kCutWords; i += kSampThreads) H[i] = 0;
    __syncthreads();
    und.each(a, w, row, h, look, lo, hi, [&](uint32_t k, uint64_t f, uint32_t n, int) {
      atomicAdd((unsigned long long*)&Hc[(k - lo) >> shift], (unsigned long long)(MASS ? f * n : n));
    });
    __syncthreads();
    if (t < 64) {  // four ranges per lane; suffix sums across the lanes
      uint64_t r[4] = {0, 0, 0, 0};
#pragma unroll
      for (int c = 0; c < kCutCopies; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] += H[c * kCutStride + 4 * lane + j];
      const uint64_t pre = wave_prefix(r[0] + r[1] + r[2] + r[3]);
      uint64_t cum = (MASS ? rest : 0) + wave_last(pre) - pre;  // above this lane's ranges
      int at = -1;
      uint64_t above = 0;
#pragma unroll
      for (int j = 3; j >= 0; --j) {
        if (MASS ? cum < thr : (cum < rest && rest <= cum + r[j])) {
          at = 4 * lane + j;
          above = cum;
        }
        cum += r[j];
      }
      // masses: of the ranges that qualify the lowest, in the lowest lane with one
      const uint64_t any = __ballot(at >= 0);
      if (lane == (any ? __ffsll((long long)any) - 1 : 0)) {
        bc[0] = (uint64_t)max(at, 0);
        bc[1] = !any ? rest : (MASS ? above : rest - above);
      }
    }
    __syncthreads();
    lo += (uint32_t)bc[0] << shift;
    hi = lo + min(hi - lo, (1u << shift) - 1u);
    rest = bc[1];
    // (the next write of bc is two barriers away)
  }
  return lo;
}

// Last launch, one workgroup per row: the exact cuts among the undecided
// tokens, the kept mass of each slice, and the draw: the first index whose
// prefix of kept mass exceeds u * total.
// The tokens of the top-p boundary key share one z, so one mass f.  The
// reference's sort puts them together (in vocabulary order: a stable sort)
// and its rule keeps the j-th of them while the mass above it, A + j f, stays
// below top_p: the first n = ceil((thr - A) / f) of them (A: the mass of the
// keys above).  When n is below their count, a slice keeps those of them that
// the slices before it leave, and a token's rank among them is the slice's
// start plus the ties of the threads before it and of its own run before it;
// otherwise all of them are kept, as every key above.
template <bool K, bool P>
__global__ __launch_bounds__(kSampThreads) void samp_draw_kernel(SampArgs a) {
  __shared__ uint64_t H[K || P ? kCutWords : 1];
  __shared__ uint32_t lk[K || P ? SampUndecided::kFlat * kSampThreads : 1];
  __shared__ uint8_t ls[K || P ? SampUndecided::kFlat * kSampThreads : 1];
  __shared__ uint32_t lc[K || P ? kSampMaxBlocks : 1];
  __shared__ uint64_t bck[2], bcp[2];
  __shared__ SampTable tb;
  __shared__ uint64_t red[kSampWaves], wtot[kSampWaves];
  __shared__ float zred[4][kSampWaves];
  __shared__ uint64_t smass[kSampMaxBlocks];
  __shared__ int stie[kSampMaxBlocks];
  __shared__ int wtie[kSampWaves];
  __shared__ int found;
  const int row_i = blockIdx.y;
  const float* row = a.x + (int64_t)row_i * a.ld;
  const uint8_t* w = samp_row_ws(a);
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const SampHead h = *(const SampHead*)(w + SampRow::kHead);  // the whole head in one load
  const uint64_t base_g = ((const uint64_t*)(w + SampRow::kSum))[min(lane, a.G - 1)];
  const float split = (K || P) && t < 64 ? samp_lane_split(w) : 0.0f;
  double uf = (double)a.u[row_i];
  uf = uf < 0.0 ? 0.0 : uf;
  if (!h.valid) {
    if (t == 0) a.tokens[row_i] = -1;
    return;
  }
  if (t == 0) found = -1;
  uint32_t kth = 0, tkey = 0;
  uint64_t tf = 0;  // mass of a boundary token when only the first tn are kept
  int tn = 0;
  if constexpr (K || P) {
    if (t < kSampMaxBlocks) {
      smass[t] = 0;
      stie[t] = 0;
    }
    if (t < 64) samp_table(split, h.m, h.low, &tb);
    SampUndecided und;
    und.load(a, w, h.m, lk, ls, lc);
    const SampLook look{&tb};
    // lowest and highest undecided z, of the k-th token's bin and of the boundary's bins
    float k0 = INFINITY, k1 = -INFINITY, p0 = INFINITY, p1 = -INFINITY;
    und.each(a, w, row, h, look, 0u, ~0u, [&](uint32_t k, uint64_t, uint32_t, int) {
      const float z = samp_unkey(k);
      const int b = look.bin(z);
      if (K && b == h.kbin) {
        k0 = fminf(k0, z);
        k1 = fmaxf(k1, z);
      }
      if (P && b >= h.lo && b <= h.hi) {
        p0 = fminf(p0, z);
        p1 = fmaxf(p1, z);
      }
    });
    if constexpr (K) {
      k0 = wave_min(k0);
      k1 = wave_max(k1);
    }
    if constexpr (P) {
      p0 = wave_min(p0);
      p1 = wave_max(p1);
    }
    if (lane == 0) {
      zred[0][wv] = k0;
      zred[1][wv] = k1;
      zred[2][wv] = p0;
      zred[3][wv] = p1;
    }
    __syncthreads();
    const int wl = min(lane, kSampWaves - 1);
    const bool topk = K && h.kbin >= 0;  // uniform; P: the boundary always lies in a bin
    uint64_t S = h.total;
    uint32_t ktop = 0;
    if constexpr (K) {
      if (topk) {
        ktop = samp_key(wave_max(zred[1][wl]));
        uint64_t rank = (uint64_t)h.krest;
        kth = samp_descend<false>(a, w, row, h, und, look, samp_key(wave_min(zred[0][wl])), ktop, rank, 0, H, bck);
      }
    }
    if constexpr (P) {
      if (topk) {
        uint64_t part = 0;
        und.each(a, w, row, h, look, kth, ktop, [&](uint32_t, uint64_t f, uint32_t n, int) { part += f * n; });
        S = h.kabove + samp_block_sum_u64(part, red);
      }
      uint64_t above = h.labove;
      const uint64_t thr = samp_thr(a.top_p, S);
      const uint32_t plo = samp_key(wave_min(zred[2][wl])), phi = samp_key(wave_max(zred[3][wl]));
      tkey = samp_descend<true>(a, w, row, h, und, look, max(plo, kth), phi, above, thr, H, bcp);
      // the tokens of the boundary key per slice, and how many of them the rule keeps
      und.each(a, w, row, h, look, tkey, tkey, [&](uint32_t, uint64_t, uint32_t n, int g) { atomicAdd(&stie[g], (int)n); });
      __syncthreads();
      const uint64_t ties = wave_total((uint32_t)stie[lane]);
      const uint64_t f0 = samp_efix(samp_unkey(tkey), h.m), need = thr - above;
      if (ties > 1 && f0 && thr > above && need < ties * f0) {
        // ceil(need / f0) <= ties: the double estimate is corrected by at most one either way
        uint64_t n = (uint64_t)ceil((double)need / (double)f0);
        if (n > 0 && (n - 1) * f0 >= need) --n;
        if (n * f0 < need) ++n;
        if (n < ties) {
          tf = f0;
          tn = (int)n;
        }
      }
    }
    // the kept mass of each slice's undecided tokens: those from the cut up
    // (boundary ties apart while tf is set)
    const uint32_t lim = max(kth, tkey);
    und.each(a, w, row, h, look, lim, ~0u, [&](uint32_t k, uint64_t f, uint32_t n, int g) {
      if (!(tf && k == tkey)) atomicAdd((unsigned long long*)&smass[g], (unsigned long long)(f * n));
    });
  }
  __syncthreads();
  const uint32_t lim = max(kth, tkey);
  // every wave: the ties before each slice (lane) and those it keeps ...
  int tbefore_g = 0, tkeep_g = 0;
  if (P && tf) {
    const int tc_g = stie[lane];
    tbefore_g = (int)wave_prefix((uint32_t)tc_g) - tc_g;
    tkeep_g = min(max(tn - tbefore_g, 0), tc_g);
  }
  // ... the slice masses, their inclusive prefix, the total
  uint64_t mine_g = lane < a.G ? base_g + tf * (uint64_t)tkeep_g : 0;
  if constexpr (K || P) mine_g += smass[lane];
  const uint64_t pre_g = wave_prefix(mine_g);
  const uint64_t total = wave_last(pre_g);
  uint64_t target = (uint64_t)(uf * (double)total);
  if (target >= total) target = total - 1;  // u = 1 (outside [0, 1)) takes the last kept token
  // the slice whose prefix first exceeds the target (the last slice at the latest)
  const uint64_t over = __ballot(lane < a.G && pre_g > target);
  const int g = over ? __ffsll((long long)over) - 1 : a.G - 1;
  const int i0 = g * a.per, i1 = min(i0 + a.per, a.V);
  const int e = (i1 - i0 + kSampThreads - 1) / kSampThreads;  // consecutive tokens per thread
  const int t0 = i0 + t * e, t1 = min(t0 + e, i1);
  float x[kSampUnroll];
#pragma unroll
  for (int j = 0; j < kSampUnroll; ++j) x[j] = row[min(t0 + j, a.V - 1)];
  target -= __shfl(pre_g - mine_g, g);  // within slice g
  const int trank0 = __shfl(tbefore_g, g);
  const float m = h.m;
  // this thread's run: the mass of its kept tokens other than split ties, and its ties
  uint64_t mine = 0;
  uint32_t myt = 0;
  const auto add = [&](float z) {
    const uint32_t key = samp_key(z);
    if (P && tf && key == tkey)
      ++myt;
    else if (key >= lim)
      mine += samp_efix(z, m);
  };
#pragma unroll
  for (int j = 0; j < kSampUnroll; ++j)  // its first tokens, loaded together
    if (t0 + j < t1) add(x[j] / a.T);
  for (int i = t0 + kSampUnroll; i < t1; ++i) add(samp_z(a, row, i));
  int rank0 = 0;  // rank of this run's first boundary tie
  if (P && tf) {  // uniform
    const int tincl = (int)wave_prefix(myt);
    if (lane == 63) wtie[wv] = tincl;
    __syncthreads();
    int tbase = trank0;
    for (int i = 0; i < wv; ++i) tbase += wtie[i];
    rank0 = tbase + tincl - (int)myt;
    mine += tf * (uint64_t)min(max(tn - rank0, 0), (int)myt);  // its ties below rank tn
  }
  // inclusive scan within the wave, then the wave totals in wave order
  uint64_t incl = wave_prefix(mine);
  if (lane == 63) wtot[wv] = incl;
  __syncthreads();
  const uint64_t wl = wave_prefix(lane < kSampWaves ? wtot[lane] : (uint64_t)0);
  if (wv > 0) incl += __shfl(wl, wv - 1);
  const uint64_t excl = incl - mine;
  if (excl <= target && target < incl) {
    uint64_t c = excl;
    int rank = rank0;
    for (int i = t0; i < t1; ++i) {
      const float z = samp_z(a, row, i);
      const uint32_t key = samp_key(z);
      if (P && tf && key == tkey)
        c += rank++ < tn ? tf : 0;
      else if (key >= lim)
        c += samp_efix(z, m);
      if (c > target) {
        found = i;
        break;
      }
    }
  }
  __syncthreads();
  if (t == 0) a.tokens[row_i] = found;
}

int64_t sample_workspace_bytes(int64_t M) { return M * SampRow::kBytes; }

namespace {

template <bool K, bool P>
void launch_sample(const SampArgs& a, int64_t M, hipStream_t st) {
  const dim3 grid((unsigned)a.G, (unsigned)M), block(kSampThreads);
  hipLaunchKernelGGL(samp_max_kernel, grid, block, 0, st, a);
  if constexpr (K || P) hipLaunchKernelGGL((samp_bins_kernel<K, P>), grid, block, 0, st, a);
  hipLaunchKernelGGL((samp_list_kernel<K, P>), grid, block, 0, st, a);
  hipLaunchKernelGGL((samp_draw_kernel<K, P>), dim3(1, (unsigned)M), block, 0, st, a);
}

}  // namespace

int launch_sample_rows(const float* x, int64_t M, int64_t V, int64_t ld, float T, int64_t top_k, float top_p,
                       const float* u, int64_t* tokens, void* ws, hipStream_t st) {
  SampArgs a{};
  a.x = x;
  a.ld = ld;
  a.V = (int)V;
  a.G = (int)((V + 2047) / 2048);
  if (a.G > kSampMaxBlocks) a.G = kSampMaxBlocks;
  a.per = (int)((V + a.G - 1) / a.G);
  a.T = T;
  a.k = top_k > 0 && top_k < V ? (int)top_k : 0;
  a.top_p = top_p > 0.0f && top_p < 1.0f ? (double)top_p : 0.0;
  a.ws = (uint8_t*)ws;
  a.u = u;
  a.tokens = tokens;
  if (a.k && a.top_p > 0.0)
    launch_sample<true, true>(a, M, st);
  else if (a.k)
    launch_sample<true, false>(a, M, st);
  else if (a.top_p > 0.0)
    launch_sample<false, true>(a, M, st);
  else
    launch_sample<false, false>(a, M, st);
  return check_launch();
}

}  // namespace sbq
