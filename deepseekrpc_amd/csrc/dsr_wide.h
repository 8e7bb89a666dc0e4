// Sliced path for FP32 and bf16 rows (gfx950, wave64): a row spread over the
// whole chip instead of walked by one workgroup.
//
// It takes every row of SamplingPolicy.probabilities (sampling.py:48-106)
// that is greedy, cuts to 1 <= top_k <= 1,024, or keeps the whole vocabulary
// (top-p, min-p, both or neither), with or without a token history, a logit
// bias, an allow mask and a tentative prefix, whatever the vocabulary size
// and row alignment.  Two to six launches, ordered by
// their boundaries (the caller's hints leave out those no row needs):
//
//   k_wide_scan     one workgroup per 8,192-token slice reads the slice once:
//                   validity, the slice's maximum and first index; the
//                   touched tokens (history, prefix, bias), whose float64
//                   adjusted values go to the row's workspace.  Top-k rows:
//                   the 16-bit key prefix of every 16-token group's maximum.
//                   Whole rows: sum exp((v - m) / T) in float64 and the mass
//                   per 1,024 bins of m - v, relative to the slice's own
//                   maximum m (the row's is not known yet).
//   k_wide_bracket  one workgroup per whole row: the row's maximum and sum, and
//                   from the slices' bin masses the values between which
//                   the min-p and top-p boundaries lie.
//   k_wide_collect  filtered whole rows: each slice lists its tokens between
//                   those values and sums the tokens above them.
//   k_wide_topk     one workgroup per top-k row: the k-th largest group
//                   prefix bounds the k-th largest token from below (the
//                   groups and touched tokens partition the row), only the
//                   groups that reach it are read again, and the few tokens
//                   above it finish on the FP32 top-k kernel's tail.
//   k_wide_draw     one workgroup per whole row: the boundary among the listed
//                   tokens by value and index as the reference's stable sort
//                   orders them (:97-102), the slice that holds u * total,
//                   and that slice's tokens in index order.
//   k_wide_probs    whole rows whose probabilities are asked for.
//
// What bounds them, at V = 129,280 (64 bf16 rows, top-k 50, 4,096-token
// histories, and 32 FP32 rows of mixed whole policies with distributions): the
// scan of top-k rows a copy's rate (12.6 us), of whole rows the float64 exps
// and LDS atomics (13.3 us); the bracket two round trips to memory (8.1 us);
// the collect its second read of the row (10.9 us); the finishing workgroups
// their chains of dependent reductions (top-k 15.5 us, draw 23.8 us); the
// probabilities their stores (14.7 us).  Before it, one workgroup per row took
// 1,013 us for the first, now 28; the split path 297 for the second, more
// (426 to 444) where it handed rows over, now 70.
//
// Bin masses only bracket a boundary (they carry 36-bit fixed point and
// FP32 rounding, and the bracket allows for both); every decision is made
// again in float64 from the listed tokens' own exps and float64 sums, in a
// fixed order.  Rows outside these limits (and invalid ones, whose status
// the reference's order decides) take the general path in the finishing
// workgroup.
#pragma once

#include "dsr_f32.h"
#include "dsr_full.h"
#include "dsr_general.h"

namespace dsr {

constexpr int kWideThreads = 256;
constexpr int kWideWaves = kWideThreads / 64;
constexpr int kWidePer = 32;                              // tokens per thread
constexpr int kWideSlice = kWideThreads * kWidePer;       // 8,192
constexpr int kWideMaxSlices = 16;
constexpr int kWideGroup = 16;                            // tokens per group maximum
constexpr int kWideGroups = kWideSlice / kWideGroup;      // 512 per slice
constexpr int kWideBins = 1024;                           // bins of (maximum - value)
constexpr int kWideCand = 2048;                           // listed tokens per slice, at most (WideLayout::cand_cap)
constexpr int kWideFine = kThreads;                       // tokens of the cut's sub-bin, resolved exactly (one per thread)
constexpr int kWidePrefix = DSR_MAX_DRAFTS;               // touched places of a tentative prefix
constexpr int kWideHistCopies = 2;
static_assert((int64_t)kWideMaxSlices * kWideSlice >= DSR_MAX_VOCAB, "the slices cover the vocabulary");
static_assert(kWideMaxSlices == kWaves, "one wave of the finishing workgroup per slice");

constexpr uint32_t kWideBad = 1u;      // NaN or +inf, or a history / bias entry the general path rejects

struct WideRec {      // one slice, from k_wide_scan
  double m;           // largest adjusted value (-inf: none)
  double sum;         // whole rows: sum exp((v - m) / T)
  double vmin;        // whole rows with no filter: a lower bound of the finite adjusted values
  long long csum;     // history counts
  int32_t first;      // greedy rows: first index holding m
  uint32_t flags;
  int32_t e0, e1;     // history entries of the slice
  int32_t b0, b1;     // bias entries of the slice
  int32_t npos;       // whole rows with no filter: finite tokens
  int32_t pad;
};
static_assert(sizeof(WideRec) == 64, "workspace layout");

struct WideSum {      // one slice, from k_wide_collect
  double kept;        // mass of the tokens certainly kept, relative to the row maximum
  double mid;         // with min-p: mass of those it keeps and top-p certainly removes
  int32_t npos;       // positive masses in `kept`
  int32_t ncand;      // listed tokens, or more than the list holds
};

struct WideRow {      // one row, from k_wide_bracket
  double M;           // row maximum
  double S;           // whole rows: sum exp((v - M) / T)
  double vmin;
  int32_t first;      // greedy rows: first index holding M
  int32_t npos;       // whole rows with no filter: finite tokens
  int32_t bad;        // invalid: the general path reports it
  int32_t pad;
  double hi, plo, phi, mlo, mhi;  // WideBracket
};

struct WideDec {      // one whole row's kept set, from k_wide_draw
  double Sk, vc;      // kept mass, value of the last kept token
  int32_t ic;         // tokens equal to vc are kept up to this index
  int32_t done;       // 0: k_wide_probs writes the row's probabilities
};

static_assert(sizeof(WideRow) <= 128 && sizeof(WideDec) <= 64, "workspace layout");

// Per-row workspace: every part a multiple of 16 bytes.  After the records
// come a top-k row's group keys, or another row's bin masses and lists, and in
// the rest its touched tokens (TOP: a top-k row's).
struct WideLayout {
  int64_t V;
  int nS;
  __host__ __device__ explicit WideLayout(int64_t vocab) : V(vocab), nS((int)((vocab + kWideSlice - 1) / kWideSlice)) {}
  // Short rows list fewer tokens per slice, to leave room for touched ones.
  __host__ __device__ int cand_cap() const { return V >= 4 * kWideSlice ? kWideCand : kWideCand / 2; }
  __host__ __device__ size_t sum_off() const { return (size_t)nS * sizeof(WideRec); }
  __host__ __device__ size_t dec_off() const { return sum_off() + (((size_t)nS * sizeof(WideSum) + 15) & ~(size_t)15); }
  __host__ __device__ size_t row_off() const { return dec_off() + 64; }
  __host__ __device__ size_t scale_off() const { return row_off() + 128; }
  __host__ __device__ size_t kind_off() const { return scale_off() + 128; }
  __host__ __device__ size_t cand_off() const { return kind_off() + (size_t)nS * kWideBins * sizeof(float); }
  template <bool TOP>
  __device__ __forceinline__ size_t touch_off() const {
    return TOP ? kind_off() + (size_t)nS * kWideGroups * sizeof(uint16_t) : cand_off() + (size_t)nS * cand_cap() * 12;
  }
  // Touched tokens it holds: a float64 value and, in a top-k row, a 16-bit key each.
  template <bool TOP>
  __device__ __forceinline__ int touch_cap() const {
    const uint32_t left = (uint32_t)(ws_stride(V) * sizeof(double) - touch_off<TOP>());  // positive from kWideMinVocab on
    return (int)((left / (TOP ? 10u : 8u)) & ~7u);
  }
  __device__ __forceinline__ WideRec* rec(char* w) const { return (WideRec*)w; }
  __device__ __forceinline__ WideSum* sum(char* w) const { return (WideSum*)(w + sum_off()); }
  __device__ __forceinline__ WideDec* dec(char* w) const { return (WideDec*)(w + dec_off()); }
  __device__ __forceinline__ WideRow* row(char* w) const { return (WideRow*)(w + row_off()); }
  __device__ __forceinline__ double* scale(char* w) const { return (double*)(w + scale_off()); }  // each slice's exp((m - M) / T)
  __device__ __forceinline__ float* hist(char* w) const { return (float*)(w + kind_off()); }
  __device__ __forceinline__ uint16_t* group(char* w) const { return (uint16_t*)(w + kind_off()); }
  // Listed tokens of slice s: values, then token ids.
  __device__ __forceinline__ double* cand_v(char* w, int s) const { return (double*)(w + cand_off()) + (size_t)s * cand_cap(); }
  __device__ __forceinline__ int32_t* cand_i(char* w, int s) const {
    return (int32_t*)(w + cand_off() + (size_t)nS * cand_cap() * 8) + (size_t)s * cand_cap();
  }
  template <bool TOP>
  __device__ __forceinline__ double* tv(char* w) const { return (double*)(w + touch_off<TOP>()); }
  __device__ __forceinline__ uint16_t* tk(char* w) const {
    return (uint16_t*)(w + touch_off<true>() + (size_t)touch_cap<true>() * 8);
  }
};

// Vocabularies the path takes: below it a row fits few slices, and the
// workspace row must hold a useful number of touched tokens.
constexpr int64_t kWideMinVocab = 8192;

enum WideKind { kWideNone = 0, kWideGreedy = 1, kWideTopK = 2, kWideWhole = 3 };

// What the path does with a row (uniform; from its policy and table sizes alone).
__device__ __forceinline__ WideKind wide_kind(const RowSpec& r, const WideLayout& L) {
  const dsr_policy_t& p = r.pol;
  if (!policy_ok(p)) return kWideNone;
  const bool top = p.temperature != 0.0 && p.top_k >= 1 && p.top_k < r.V;
  if (r.pen_n < 0 || r.bias_n < 0 || r.pen_n + r.bias_n + kWidePrefix > (top ? L.touch_cap<true>() : L.touch_cap<false>()))
    return kWideNone;
  if (p.temperature == 0.0) return kWideGreedy;
  if (top) return p.top_k <= kSplitMaxK ? kWideTopK : kWideNone;
  return p.temperature >= 1e-290 ? kWideWhole : kWideNone;  // 1 / T stays finite
}

__device__ __forceinline__ bool wide_nofilter(const dsr_policy_t& p) { return !(p.top_p < 1.0) && p.min_p == 0.0; }

// Penalties that leave every logit as it is.
__device__ __forceinline__ bool wide_neutral(const dsr_policy_t& p) {
  return p.repetition_penalty == 1.0 && p.presence_penalty == 0.0 && p.frequency_penalty == 0.0;
}

// Why a row is outside the path.
__device__ __forceinline__ int wide_outside(const RowSpec& r) {
  if (!policy_ok(r.pol)) return kHandPolicy;
  return r.pol.top_k > kSplitMaxK && r.pol.top_k < r.V ? kHandTopK : kHandCapacity;
}

__device__ __forceinline__ bool wide_touched(const RowSpec& r) { return r.pen_n > 0 || r.prefix_n > 0 || r.bias_n > 0; }

// ---------------------------------------------------------------------------
// Loads.  16 bytes at any element alignment (the row may start anywhere).

struct __attribute__((packed, aligned(4))) WideQ4 { uint32_t w[4]; };
struct __attribute__((packed, aligned(2))) WideQ2 { uint32_t w[4]; };

// Index of a thread's k-th token of a slice: 16-byte vectors, consecutive
// threads on consecutive vectors.
template <int DT>
__device__ __forceinline__ int64_t wide_index(int64_t lo, int t, int k) {
  constexpr int W = DT == DSR_BF16 ? 8 : 4;
  return lo + (int64_t)(k / W) * (W * kWideThreads) + (int64_t)t * W + (k % W);
}

// This thread's 32 tokens of the slice at lo as floats; tokens past the row
// become -inf.  Vectors wholly inside the row are read whole, a last partial
// one token by token.
template <int DT>
__device__ __forceinline__ void wide_load(const RowSpec& r, int64_t lo, int t, float v[kWidePer]) {
  constexpr int W = DT == DSR_BF16 ? 8 : 4;
#pragma unroll
  for (int q = 0; q < kWidePer / W; ++q) {
    const int64_t i = wide_index<DT>(lo, t, q * W);
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    if (i + W <= r.V) {
      if constexpr (DT == DSR_BF16) {
        const WideQ2 x = *(const WideQ2*)((const uint16_t*)r.logits + i);
        w[0] = x.w[0]; w[1] = x.w[1]; w[2] = x.w[2]; w[3] = x.w[3];
      } else {
        const WideQ4 x = *(const WideQ4*)((const float*)r.logits + i);
        w[0] = x.w[0]; w[1] = x.w[1]; w[2] = x.w[2]; w[3] = x.w[3];
      }
    } else {
#pragma unroll
      for (int e = 0; e < W; ++e) {
        const bool in = i + e < r.V;
        if constexpr (DT == DSR_BF16) {
          const uint32_t b = in ? (uint32_t)((const uint16_t*)r.logits)[i + e] : 0xFF80u;
          w[e >> 1] |= b << (16 * (e & 1));
        } else {
          w[e] = in ? ((const uint32_t*)r.logits)[i + e] : 0xFF800000u;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < W; ++e)
      v[q * W + e] = DT == DSR_BF16 ? __uint_as_float(((w[e >> 1] >> (16 * (e & 1))) & 0xFFFFu) << 16) : __uint_as_float(w[e]);
  }
}

// Bit k set when this thread's k-th token is allowed (tokens past the row: unspecified).
template <int DT>
__device__ __forceinline__ uint32_t wide_allowed(const RowSpec& r, int64_t lo, int t) {
  if (!r.allow) return 0xFFFFFFFFu;
  constexpr int W = DT == DSR_BF16 ? 8 : 4;
  uint32_t m = 0u;
#pragma unroll
  for (int q = 0; q < kWidePer / W; ++q) {
    const int64_t i = wide_index<DT>(lo, t, q * W);  // a multiple of W: one word holds the vector's bits
    const uint32_t w = i < r.V ? r.allow[i >> 5] : 0u;
    m |= ((w >> (i & 31)) & ((1u << W) - 1u)) << (q * W);
  }
  return m;
}

// The same for an LDS bitmap of the slice's tokens.
template <int DT>
__device__ __forceinline__ uint32_t wide_bits(const uint32_t* bm, int t) {
  constexpr int W = DT == DSR_BF16 ? 8 : 4;
  uint32_t m = 0u;
#pragma unroll
  for (int q = 0; q < kWidePer / W; ++q) {
    const int i = (int)wide_index<DT>(0, t, q * W);
    m |= ((bm[i >> 5] >> (i & 31)) & ((1u << W) - 1u)) << (q * W);
  }
  return m;
}

// FP32 bits of the four tokens from i (a multiple of 4) on; those past the row are -inf.
template <int DT>
__device__ __forceinline__ void wide_quad(const RowSpec& r, int64_t i, uint32_t w[4]) {
  if (i + 4 <= r.V) {
    if constexpr (DT == DSR_BF16) {
      struct __attribute__((packed, aligned(2))) Q { uint32_t w[2]; };
      const Q x = *(const Q*)((const uint16_t*)r.logits + i);
      w[0] = x.w[0] << 16;
      w[1] = x.w[0] & 0xFFFF0000u;
      w[2] = x.w[1] << 16;
      w[3] = x.w[1] & 0xFFFF0000u;
    } else {
      const WideQ4 x = *(const WideQ4*)((const float*)r.logits + i);
      w[0] = x.w[0]; w[1] = x.w[1]; w[2] = x.w[2]; w[3] = x.w[3];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = i + e < r.V;
      if constexpr (DT == DSR_BF16) w[e] = in ? (uint32_t)((const uint16_t*)r.logits)[i + e] << 16 : 0xFF800000u;
      else w[e] = in ? ((const uint32_t*)r.logits)[i + e] : 0xFF800000u;
    }
  }
}

// ---------------------------------------------------------------------------
// Touched tokens.

// Entries [e0, e1) of the sorted list ids[0, n) that lie in [lo, hi): each
// wave narrows both bounds by 128 probes a round (two rounds up to 16,384
// entries), without a barrier.  For a list that is not sorted the result is
// some range inside [0, n]; wide_row_of sees such a list by the slices'
// ranges not meeting, or by an entry outside its slice.
__device__ __forceinline__ void wide_range(const int32_t* ids, int n, int lo, int hi, int& e0, int& e1) {
  const int l = lane_id();
  int a0 = 0, n0 = n, a1 = 0, n1 = n;  // the bound lies in [a, a + n]
  while (n0 > 0 || n1 > 0) {           // uniform; n shrinks at least by half each round
    const int s0 = (n0 + 127) >> 7, s1 = (n1 + 127) >> 7;
    int c0 = 0, c1 = 0;
    int32_t x[4];
    bool in[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = ((q & 1) * 64 + l + 1) * (q < 2 ? s0 : s1) - 1;
      in[q] = i >= 0 && i < (q < 2 ? n0 : n1);
      x[q] = in[q] ? ids[(q < 2 ? a0 : a1) + i] : 0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = (int)__popcll(__ballot(in[q] && x[q] < (q < 2 ? lo : hi)));
      if (q < 2) c0 += c; else c1 += c;
    }
    const int r0 = n0 - c0 * s0, r1 = n1 - c1 * s1;  // entries not below the last probe passed
    a0 += c0 * s0;
    a1 += c1 * s1;
    n0 = r0 < s0 - 1 ? r0 : s0 - 1;
    n1 = r1 < s1 - 1 ? r1 : s1 - 1;
    if (n0 < 0) n0 = 0;
    if (n1 < 0) n1 = 0;
  }
  e0 = a0;
  e1 = a1 < a0 ? a0 : a1;  // an unsorted list may order the bounds either way
}

// Position of id in the sorted list ids[lo, hi), or -1.
__device__ __forceinline__ int wide_find(const int32_t* ids, int lo, int hi, int32_t id) {
  const int end = hi;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (ids[mid] < id) lo = mid + 1; else hi = mid;
  }
  return lo < end && ids[lo] == id ? lo : -1;
}

// Visits this thread's touched places of a slice: place (index into tv) and
// token.  A place whose token is counted at another place holds -inf.
template <int STRIDE, class F>
__device__ __forceinline__ void wide_touched_each(const RowSpec& r, int e0, int e1, int b0, int b1, int64_t lo, int64_t hi,
                                                  F f) {
  for (int e = e0 + (int)threadIdx.x; e < e1; e += STRIDE) f(e, r.pen_ids[e]);
  if ((int)threadIdx.x < r.prefix_n) {
    const int32_t id = r.prefix[threadIdx.x];
    if (id >= lo && id < hi) f((int)r.pen_n + (int)threadIdx.x, id);
  }
  for (int b = b0 + (int)threadIdx.x; b < b1; b += STRIDE) f((int)r.pen_n + kWidePrefix + b, r.bias_ids[b]);
}

// The largest float not above v.
__device__ __forceinline__ float wide_floor(double v) {
  float f = (float)v;
  if ((double)f > v) {  // step one float down
    uint32_t b = __float_as_uint(f);
    if (f > 0.0f) b -= 1u;
    else if (f == 0.0f) b = 0x80000001u;
    else b += 1u;
    f = __uint_as_float(b);
  }
  return f;
}

// Its order key (finite v), as f32_key orders floats.
__device__ __forceinline__ uint32_t wide_floor_key(double v) { return f32_key(__float_as_uint(wide_floor(v)), true); }

// The float an order key (f32_key) stands for.
__device__ __forceinline__ float wide_key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// Bins per logit: a whole row's masses are counted by (maximum - value), as its
// law depends on that alone, in bins of T / 32, or sqrt(T) / 32 above T = 1
// (of T / 32 a hot row would fill few).  So 1,024 bins reach 32 nats down, where
// a token's mass is 1e-14, and 32 / sqrt(T) nats in hot rows, whose logits
// span fewer; what lies lower shares the last bin.
__device__ __forceinline__ double wide_per_logit(const dsr_policy_t& p) {
  const double T = fmax(p.temperature, 1e-6);
  return 32.0 / (T > 1.0 ? sqrt(T) : T);
}

// The bin of distance y (in bins, >= 0; a NaN: the last).
__device__ __forceinline__ int wide_bin(double y) { return (int)fmin(y, (double)(kWideBins - 1)); }

// a / T, rounded as the IEEE quotient (sampling.py:88 divides), from iT = 1 / T
// rounded: a product and one correction by its exact remainder (P. W.
// Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", IBM J. Res. Dev. 34(1), 1990).  Minus infinity, and a product
// that overflows to it, give a NaN; wide_exp takes that as minus infinity.
__device__ __forceinline__ double wide_over(double a, double T, double iT) {
  const double q = a * iT;
  return fma(fma(-q, T, a), iT, q);
}

// exp(z), z <= 0 or a NaN (0; it underflows to 0 below -745.14).  The library's
// exp, as in the general path: with it and the divide above the scan of 32 FP32
// rows takes 13.5 us, with exp_nonpos and a product by 1 / T 13.3.
__device__ __forceinline__ double wide_exp(double z) { return exp(fmax(z, -746.0)); }

// ---------------------------------------------------------------------------
// Rows of dsr_sample_rows.

__device__ __forceinline__ RowSpec sample_row_spec(const dsr_sample_args_t& a, int64_t row, double* W);

struct WideSampleRows {
  dsr_sample_args_t a;
  __device__ __forceinline__ bool takes(int64_t) const { return true; }
  __device__ __forceinline__ char* ws(int64_t d) const { return (char*)a.workspace + (size_t)d * ws_stride(a.vocab) * sizeof(double); }
  __device__ __forceinline__ RowSpec spec(int64_t d) const { return sample_row_spec(a, d, (double*)ws(d)); }
  __device__ __forceinline__ void onehot(int64_t, int64_t) const {}
  // Unfiltered rows whose table changes no logit stay on the general path, as before this one.
  __device__ __forceinline__ WideKind kind(const RowSpec& r, const WideLayout& L) const {
    const WideKind k = wide_kind(r, L);
    return k == kWideWhole && r.pen_n > 0 && wide_nofilter(r.pol) && wide_neutral(r.pol) ? kWideNone : k;
  }
};

// ---------------------------------------------------------------------------
// Step 1.

struct WideWaveRec {   // one wave's part of a slice
  double tmax;          // touched tokens
  uint32_t key, kmin;   // f32_key of the largest and smallest finite untouched value
  int32_t first, tfirst;
  uint32_t n, csum, bad, pad;
};

// A token's part of a bin's 64-bit word: the bits of the double 2^52 + 2^50
// + mass * 2^36.  A slice's masses sum below 2^50, so the low 50 bits of a
// word are their sum (the others mean nothing).
constexpr double kWideOne = 0x1p52 + 0x1p50;
struct WideHist {
  // The copies start on different banks.
  unsigned long long w[kWideHistCopies][kWideBins + 8];
};

template <bool WHOLE>
struct WideScanShared {
  struct None {};
  typename std::conditional<WHOLE, WideHist, None>::type hist;
  uint32_t tbits[kWideSlice / 32];                        // touched tokens
  uint32_t kbits[kWideSlice / 32];                        // finite tokens (kept-bit output)
  WideWaveRec wr[kWideWaves];
  double rs[kWideWaves];
  int found[kWidePrefix];
};

// probs_later: k_wide_probs writes the probability rows of whole rows.  WHOLE:
// the batch may hold whole rows.
template <class Src, int DT, bool WHOLE>
__global__ __launch_bounds__(kWideThreads) void k_wide_scan(Src src, int nS, int probs_later) {
  __shared__ WideScanShared<WHOLE> sh;
  const int t = threadIdx.x;
  const int64_t d = blockIdx.x / (unsigned)nS;
  const int s = (int)(blockIdx.x % (unsigned)nS);
  if (!src.takes(d)) return;
  const RowSpec r = src.spec(d);
  const WideLayout L(r.V);
  const WideKind kind = src.kind(r, L);
  if (kind == kWideNone || (!WHOLE && kind == kWideWhole)) return;  // the finishing workgroup's general path
  char* ws = src.ws(d);
  const int lo = s * kWideSlice, hi = lo + kWideSlice < (int)r.V ? lo + kWideSlice : (int)r.V;
  const dsr_policy_t& p = r.pol;
  const bool touched = wide_touched(r);  // uniform
  int e0 = 0, e1 = 0, b0 = 0, b1 = 0;
  if (r.pen_n > 0) wide_range(r.pen_ids, (int)r.pen_n, lo, hi, e0, e1);
  if (r.bias_n > 0) wide_range(r.bias_ids, (int)r.bias_n, lo, hi, b0, b1);

  float v[kWidePer];
  wide_load<DT>(r, lo, t, v);
  uint32_t ok = wide_allowed<DT>(r, lo, t);  // allowed and untouched

  const bool whole = WHOLE && kind == kWideWhole;
  const bool nof = wide_nofilter(p);
  const bool hist = whole && !nof;  // only filtered rows look for a bin
  if (t < kWideSlice / 32) {
    sh.tbits[t] = 0u;
    sh.kbits[t] = 0u;
  }
  if (t < kWidePrefix) sh.found[t] = 0;
  if constexpr (WHOLE) {
    if (hist) {
      uint4* z = (uint4*)&sh.hist;
      for (int b = t; b < (int)(sizeof(sh.hist) / 16); b += kWideThreads) z[b] = make_uint4(0u, 0u, 0u, 0u);
    }
  }

  uint32_t bad = 0u;
  double tmax = -INFINITY;
  uint32_t kmin = 0xFFFFFFFFu, tn = 0u, csum = 0u;  // csum saturates: more than the limit is an error anyway
  int32_t tfirst = INT32_MAX;
  double* tv = kind == kWideTopK ? L.tv<true>(ws) : L.tv<false>(ws);
  uint16_t* tk = L.tk(ws);
  auto raw = [&](int32_t id) -> double {
    return DT == DSR_BF16 ? (double)__uint_as_float((uint32_t)((const uint16_t*)r.logits)[id] << 16)
                          : (double)((const float*)r.logits)[id];
  };
  // A touched token's part in the slice's maximum and count, and its key.
  auto settle = [&](int at, int32_t id, double x) {
    const bool fin = x > -(double)INFINITY;
    const uint32_t key = wide_floor_key(x);
    if (fin && id >= lo && id < hi) {
      if (x > tmax || (x == tmax && id < tfirst)) {
        tmax = x;
        tfirst = id;
      }
      kmin = min(kmin, key);
      ++tn;
      if (r.kept_bits) atomicOr(&sh.kbits[(id - lo) >> 5], 1u << ((id - lo) & 31));
    }
    if (kind == kWideTopK) tk[at] = fin ? (uint16_t)(key >> 16) : (uint16_t)0;
  };
  // Values of the thread's first kKeep history entries stay in registers when
  // nothing else can change them.
  constexpr int kKeep = 4;
  const bool simple = r.prefix_n == 0 && r.bias_n == 0;
  double keep[kKeep];
#pragma unroll
  for (int i = 0; i < kKeep; ++i) keep[i] = -INFINITY;
  if (touched) {
    lds_barrier();  // the bitmaps are clear
    // Penalties (sampling.py:59-66) in the general path's float64 order, the
    // mask after them (-inf is a fixed point of both), and the table checks
    // of :55-58, :62-65 for the slice's own entries.
    auto entry = [&](int e) -> double {
      const int32_t id = r.pen_ids[e];
      const int32_t prv = e > e0 ? r.pen_ids[e - 1] : -1;
      long long c = r.pen_count[e], g = r.pen_gen[e];
      const bool in = id >= lo && id < hi && prv < id;
      int pre = 0;
      for (int q = 0; q < r.prefix_n; ++q)
        if (r.prefix[q] == id) {
          ++pre;
          sh.found[q] = 1;
        }
      if (!in || c < 0) bad = 1u;
      c += pre;
      g += pre;
      if (c > DSR_MAX_COUNT || g < 0 || g > c) bad = 1u;
      else csum = min(csum + (uint32_t)max(c, 0ll), 2u * DSR_MAX_COUNT);
      double x = -INFINITY;
      if (in) {
        atomicOr(&sh.tbits[(id - lo) >> 5], 1u << ((id - lo) & 31));
        x = raw(id);
        if (c > 0) x = x >= 0.0 ? x / p.repetition_penalty : x * p.repetition_penalty;
        x -= p.presence_penalty * (g > 0 ? 1.0 : 0.0) + p.frequency_penalty * (double)g;
        if (!allowed_bit(r.allow, id)) x = -INFINITY;
        if (!(x == x)) x = -INFINITY;  // a NaN logit: the row is invalid
      }
      tv[e] = x;
      if (simple) settle(e, id, x);
      return x;
    };
#pragma unroll
    for (int i = 0; i < kKeep; ++i) {
      const int e = e0 + t + i * kWideThreads;
      if (e < e1) keep[i] = entry(e);
    }
    for (int e = e0 + t + kKeep * kWideThreads; e < e1; e += kWideThreads) entry(e);
    if (!simple) {
      __syncthreads();  // found[], the history's bits and values
      if (t < r.prefix_n) {  // prefix tokens that the table does not hold
        const int32_t id = r.prefix[t];
        if (id < 0 || id >= r.V) bad = 1u;
        if (id >= lo && id < hi) {
          double x = -INFINITY;
          if (!sh.found[t]) {
            int c = 0;
            bool first = true;
            for (int q = 0; q < r.prefix_n; ++q) {
              c += r.prefix[q] == id ? 1 : 0;
              if (q < t && r.prefix[q] == id) first = false;
            }
            csum += 1;
            if (first) {
              x = raw(id);
              x = x >= 0.0 ? x / p.repetition_penalty : x * p.repetition_penalty;
              x -= p.presence_penalty * 1.0 + p.frequency_penalty * (double)c;
              if (!allowed_bit(r.allow, id)) x = -INFINITY;
              if (!(x == x)) x = -INFINITY;
              atomicOr(&sh.tbits[(id - lo) >> 5], 1u << ((id - lo) & 31));
            }
          }
          tv[r.pen_n + t] = x;
        }
      }
      __syncthreads();
      // Bias (sampling.py:69-74): added to a touched token where it stands,
      // else the token's own place.  Ids are unique, so each bit tested here is
      // set by this thread alone.
      for (int b = b0 + t; b < b1; b += kWideThreads) {
        const int32_t id = r.bias_ids[b];
        const double bv = r.bias_val[b];
        double x = -INFINITY;
        if (!(id >= lo && id < hi) || (b > b0 && r.bias_ids[b - 1] >= id) || !(bv >= -100.0 && bv <= 100.0)) {
          bad = 1u;
        } else if ((sh.tbits[(id - lo) >> 5] >> ((id - lo) & 31)) & 1u) {
          int at = wide_find(r.pen_ids, e0, e1, id);
          for (int q = 0; at < 0 && q < r.prefix_n; ++q)
            if (r.prefix[q] == id) at = (int)r.pen_n + q;  // the first occurrence holds the value
          if (at >= 0) tv[at] += bv;
          else bad = 1u;  // an unsorted table
        } else {
          x = raw(id) + bv;
          if (!allowed_bit(r.allow, id)) x = -INFINITY;
          if (!(x == x)) x = -INFINITY;
          atomicOr(&sh.tbits[(id - lo) >> 5], 1u << ((id - lo) & 31));
        }
        tv[r.pen_n + kWidePrefix + b] = x;
      }
      __syncthreads();
      wide_touched_each<kWideThreads>(r, e0, e1, b0, b1, lo, hi, [&](int at, int32_t id) { settle(at, id, tv[at]); });
    }
    lds_barrier();  // the touched bits
    ok &= ~wide_bits<DT>(sh.tbits, t);
  }

  // The thread's own tokens: validity (:50-52; masked tokens included; x * 0
  // is NaN for NaN and infinities, and -inf is allowed), then masked and
  // touched tokens become -inf, and the maximum.
  {
    float z = 0.0f;
#pragma unroll
    for (int k = 0; k < kWidePer; ++k) z = __builtin_fmaf(v[k], 0.0f, z);
    if (__ballot(z != z)) {  // uniform over the wave
#pragma unroll
      for (int k = 0; k < kWidePer; ++k) bad |= __builtin_isfpclass(v[k], 0x0203) ? 1u : 0u;  // NaN or +inf
    }
  }
  if (r.allow || touched) {  // uniform
#pragma unroll
    for (int k = 0; k < kWidePer; ++k) {
      const uint32_t am = (uint32_t)((int32_t)(ok << (31 - k)) >> 31);
      v[k] = __uint_as_float((__float_as_uint(v[k]) & am) | (0xFF800000u & ~am));
    }
  }
  float m = v[0];
#pragma unroll
  for (int k = 1; k < kWidePer; ++k) m = fmaxf(m, v[k]);  // NaN: the row is invalid
  const uint32_t key = m > -INFINITY ? f32_key(__float_as_uint(m), true) : 0u;
  int mk = 0;
  if (kind == kWideGreedy) {  // the first index holding it
#pragma unroll
    for (int k = kWidePer - 1; k >= 0; --k) mk = v[k] == m ? k : mk;
  }
  if (whole && nof) {  // read for these rows alone
    uint32_t c = 0u;
    float mn = INFINITY;
#pragma unroll
    for (int k = 0; k < kWidePer; ++k) {
      const bool f = v[k] > -INFINITY;
      c += f ? 1u : 0u;
      mn = fminf(mn, f ? v[k] : INFINITY);
    }
    tn += c;
    if (c) kmin = min(kmin, f32_key(__float_as_uint(mn), true));
  }
  if (r.kept_bits && whole) {  // whole rows keep every finite token
    if (!touched) lds_barrier();  // every word is clear (uniform; touched rows have passed theirs)
    constexpr int W = DT == DSR_BF16 ? 8 : 4;
#pragma unroll
    for (int q = 0; q < kWidePer / W; ++q) {
      const int i = (int)wide_index<DT>(0, t, q * W);
      uint32_t f = 0u;
#pragma unroll
      for (int e = 0; e < W; ++e) f |= v[q * W + e] > -INFINITY ? 1u << e : 0u;
      if (f) atomicOr(&sh.kbits[i >> 5], f << (i & 31));
    }
  }
  // One barrier for every reduction: each wave's results, then all of them by every thread.
  {
    WideWaveRec w;
    w.key = wave_reduce_dpp(key, OpMax());
    w.first = INT32_MAX;
    if (kind == kWideGreedy)
      w.first = (int32_t)wave_reduce_dpp(key && key == w.key ? (uint32_t)wide_index<DT>(lo, t, mk) : (uint32_t)INT32_MAX, OpMin());
    w.kmin = 0xFFFFFFFFu;
    w.n = 0u;
    if (whole && nof) {
      w.kmin = wave_reduce_dpp(kmin, OpMin());
      w.n = wave_reduce_dpp(tn, OpSum());
    }
    w.bad = __ballot(bad != 0u) ? 1u : 0u;
    w.tmax = -INFINITY;
    w.tfirst = INT32_MAX;
    w.csum = 0u;
    w.pad = 0u;
    if (touched) {
      w.tmax = wave_reduce_dpp(tmax, OpMax());
      w.tfirst = (int32_t)wave_reduce_dpp((uint32_t)(tmax == w.tmax ? tfirst : INT32_MAX), OpMin());
      w.csum = wave_reduce_dpp(csum, OpSum());
    }
    if (lane_id() == 0) sh.wr[wave_id()] = w;
  }
  lds_barrier();
  WideRec o;
  o.sum = 0.0;
  o.csum = 0;
  o.flags = 0u;
  o.npos = 0;
  o.e0 = e0;
  o.e1 = e1;
  o.b0 = b0;
  o.b1 = b1;
  o.pad = 0;
  {
    uint32_t K = 0u, kn = 0xFFFFFFFFu;
    int32_t first = INT32_MAX, tf = INT32_MAX;
    double tm = -INFINITY;
#pragma unroll
    for (int q = 0; q < kWideWaves; ++q) {
      const WideWaveRec w = sh.wr[q];
      first = w.key > K ? w.first : (w.key == K ? min(first, w.first) : first);
      K = max(K, w.key);
      kn = min(kn, w.kmin);
      o.npos += (int32_t)w.n;
      o.flags |= w.bad ? kWideBad : 0u;
      if (touched) {
        tf = w.tmax > tm ? w.tfirst : (w.tmax == tm ? min(tf, w.tfirst) : tf);
        tm = fmax(tm, w.tmax);
        o.csum += w.csum;
      }
    }
    const double um = K ? (double)wide_key_value(K) : -(double)INFINITY;
    o.m = fmax(um, tm);
    o.first = um > tm ? first : (um < tm ? tf : min(first, tf));
    o.vmin = kn == 0xFFFFFFFFu ? (double)INFINITY : (double)wide_key_value(kn);  // touched values: the float below
  }
  const double M = o.m;

  // Outputs of the slice: kept tokens are written by the finishing steps.
  if (!(whole && probs_later)) {
    if (r.probs_f32)
      for (int i = lo + t; i < hi; i += kWideThreads) r.probs_f32[i] = 0.0f;
    if (r.probs_f64)
      for (int i = lo + t; i < hi; i += kWideThreads) r.probs_f64[i] = 0.0;
  }
  if (r.kept_bits) {
    const int64_t w = (lo >> 5) + t;
    if (t < kWideSlice / 32 && w < r.kept_words) r.kept_bits[w] = whole ? sh.kbits[t] : 0u;
  }

  if (kind == kWideTopK) {
    // 16-token group maxima: four lanes (FP32) or two (bf16) hold a group;
    // vector q of lane group j is group q * (threads / lanes) + j.
    uint16_t* g = L.group(ws) + s * kWideGroups;
    constexpr int W = DT == DSR_BF16 ? 8 : 4;
    constexpr int kLanes = kWideGroup / W;
#pragma unroll
    for (int q0 = 0; q0 < kWidePer / W; q0 += kLanes) {
      uint32_t mine = 0u;
#pragma unroll
      for (int j = 0; j < kLanes; ++j) {
        const int q = q0 + j;
        float x = v[q * W];
#pragma unroll
        for (int e = 1; e < W; ++e) x = fmaxf(x, v[q * W + e]);
        x = fmaxf(x, __uint_as_float(dpp32<0xB1>(0u, __float_as_uint(x))));
        if (kLanes == 4) x = fmaxf(x, __uint_as_float(dpp32<0x4E>(0u, __float_as_uint(x))));
        if ((t % kLanes) == j) mine = f32_key(__float_as_uint(x), true) >> 16;
      }
      g[(q0 + t % kLanes) * (kWideThreads / kLanes) + t / kLanes] = (uint16_t)mine;
    }
  }
  if constexpr (WHOLE) {
    if (whole && M > -(double)INFINITY) {
      const double iT = 1.0 / p.temperature, per = wide_per_logit(p);
      double sum = 0.0;
      unsigned long long* h = sh.hist.w[t & (kWideHistCopies - 1)];
      auto add = [&](double x) {  // x = -inf adds 0
        const double e = wide_exp(wide_over(x - M, p.temperature, iT));
        sum += e;
        // A smaller mass is 0 in these units; many such tokens share the last bin.
        if (hist && e > 0x1p-37)
          atomicAdd(&h[wide_bin((M - x) * per)], (unsigned long long)__double_as_longlong(__builtin_fma(e, 0x1p36, kWideOne)));
      };
#pragma unroll
      for (int k = 0; k < kWidePer; ++k) {
        add((double)v[k]);
        if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // four exps in flight: more cost registers
      }
      if (touched) {
        auto again = [&](double x) {
          if (x > -(double)INFINITY) add(x);
        };
        if (simple) {
#pragma unroll
          for (int i = 0; i < kKeep; ++i) again(keep[i]);
          for (int e = e0 + t + kKeep * kWideThreads; e < e1; e += kWideThreads) again(tv[e]);
        } else {
          wide_touched_each<kWideThreads>(r, e0, e1, b0, b1, lo, hi, [&](int at, int32_t) { again(tv[at]); });
        }
      }
      sum = wave_sum(sum);
      if (lane_id() == 0) sh.rs[wave_id()] = sum;
      lds_barrier();  // the sums, and the histogram
#pragma unroll
      for (int q = 0; q < kWideWaves; ++q) o.sum += sh.rs[q];
      if (hist) {
        float4* ho = (float4*)(L.hist(ws) + s * kWideBins) + t;  // bins 4t .. 4t + 3
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          unsigned long long x = 0ull;
#pragma unroll
          for (int c = 0; c < kWideHistCopies; ++c) x += sh.hist.w[c][4 * t + i];
          f[i] = (float)((double)(x & ((1ull << 50) - 1ull)) * 0x1p-36);
        }
        *ho = make_float4(f[0], f[1], f[2], f[3]);
      }
    }
  }
  if (t == 0) L.rec(ws)[s] = o;
}

// ---------------------------------------------------------------------------
// What the slices' records say about a row, in every lane (uniform).  WHOLE:
// S, lane l's factor exp((m - M) / T) of slice l, and that slice's maximum.
template <bool WHOLE>
__device__ __forceinline__ WideRow wide_row_of(const WideLayout& L, char* ws, const RowSpec& r, double& factor, double& m) {
  const int l = lane_id();
  WideRow o;
  WideRec x;
  x.m = -INFINITY;
  x.sum = 0.0;
  x.vmin = INFINITY;
  x.csum = 0;
  x.first = INT32_MAX;
  x.flags = 0u;
  x.e0 = x.e1 = x.b0 = x.b1 = x.npos = 0;
  if (l < L.nS) x = L.rec(ws)[l];
  // Slices are on lanes 0..15: one DPP row.
  o.M = lane_value(row_reduce(x.m, OpMax()), 0);
  o.first = (int32_t)lane_value(row_reduce((uint32_t)(x.m == o.M ? x.first : INT32_MAX), OpMin()), 0);
  const long long csum = lane_value(row_reduce(x.csum, OpSum()), 0);
  // The slices' entry ranges must tile the tables (they do when the ids increase).
  const int pe1 = (int)__shfl_up(x.e1, 1), pb1 = (int)__shfl_up(x.b1, 1);
  bool off = l < L.nS && (x.flags & kWideBad);
  if (l < L.nS) {
    off = off || x.e0 != (l ? pe1 : 0) || x.b0 != (l ? pb1 : 0);
    if (l == L.nS - 1) off = off || x.e1 != (int)r.pen_n || x.b1 != (int)r.bias_n;
  }
  m = x.m;
  o.bad = __ballot(off) != 0ull || csum > DSR_MAX_COUNT || !(o.M > -(double)INFINITY);
  o.S = 0.0;
  o.pad = 0;
  if constexpr (WHOLE) {
    o.vmin = lane_value(row_reduce(x.vmin, OpMin()), 0);
    o.npos = (int32_t)lane_value(row_reduce((uint32_t)x.npos, OpSum()), 0);
    factor = x.m > -(double)INFINITY ? wide_exp((x.m - o.M) / r.pol.temperature) : 0.0;
    o.S = lane_value(row_reduce(factor * x.sum, OpSum()), 0);
  }
  return o;
}

// A whole row whose positive masses the records cannot count: some finite
// token's exp may underflow.
__device__ __forceinline__ bool wide_spread(const WideRow& w, const dsr_policy_t& p) {
  return !((w.vmin - w.M) / p.temperature > -700.0);
}

// ---------------------------------------------------------------------------
// Step 2.

// The values between which the boundaries of a filtered whole row lie.  Tokens
// above `hi` are kept; those in [plo, phi] and [mlo, mhi] are listed; those
// between mhi and plo count in the min-p mass only.  V: double, or float for
// the same tests on untouched tokens.
template <class V>
struct WideBracket {
  V hi;
  V plo, phi;  // top-p (inf, -inf: none)
  V mlo, mhi;  // min-p (inf, -inf: none)
  __device__ __forceinline__ bool kept(V v) const { return v > hi; }
  __device__ __forceinline__ bool listed(V v) const {
    return (bool)(((int)(v >= plo) & (int)(v <= phi)) | ((int)(v >= mlo) & (int)(v <= mhi)));
  }
  __device__ __forceinline__ bool middle(V v) const { return (bool)((int)(v < plo) & (int)(v > mhi)); }
};

__device__ __forceinline__ WideBracket<float> wide_bracket_f(const WideBracket<double>& b) {
  return {wide_floor(b.hi), -wide_floor(-b.plo), wide_floor(b.phi), -wide_floor(-b.mlo), wide_floor(b.mhi)};
}

constexpr int kBracketThreads = kWideBins / 2;

struct WideBracketShared {
  double blk[kBracketThreads / 64];
  double pre[kWideBins];  // running mass, see wide_bracket
  double scale[kWideMaxSlices];
  int off[kWideMaxSlices];
  int b[2];
};

// Relative and absolute slack of a running bin mass: FP32 bin sums and
// 2^-36 fixed-point masses (an absolute 2^-37 per token of a row whose
// largest mass is 1).
constexpr double kWideRel = 0x1p-20;
constexpr double kWideAbs = 0x1p-18;

// Every thread of the workgroup calls.
//
// With y = (M - v) * per, a token of slice s in its bin j has y in [d + j, d + j
// + 1), d = (M - m_s) * per.  R(b) = the mass of the bins with floor(d) + j <= b
// is at least the mass of the tokens with y < b + 1, and at most that of those
// with y < b + 2.  Bins widened by a hundredth take care of the rounding of y.
__device__ __forceinline__ WideBracket<double> wide_bracket(const WideLayout& L, char* ws, const RowSpec& r, const WideRow& w,
                                                            WideBracketShared& sh) {
  const int t = threadIdx.x;
  const dsr_policy_t& p = r.pol;
  const float* h = L.hist(ws);
  const double per = wide_per_logit(p);
  constexpr int kLast = kWideBins - 2;  // the last bin has no end
  const int b0 = 2 * t;                 // this thread's bins: b0, b0 + 1
  double x0 = 0.0, x1 = 0.0;
  {
    // Slices past the row's read its last one again (a branch would make each
    // load wait for the one before).  Theirs count nothing, nor do those of a
    // slice without a finite token, which k_wide_scan leaves unwritten: a
    // factor of 0 is selected on, for what lies there may be a NaN.
    float q[kWideMaxSlices][2];
#pragma unroll
    for (int s = 0; s < kWideMaxSlices; ++s) {
      const float* hs = h + min(s, L.nS - 1) * kWideBins;
      const int j = b0 - sh.off[s];
      q[s][0] = hs[max(j, 0)];
      q[s][1] = hs[max(j + 1, 0)];
    }
#pragma unroll
    for (int s = 0; s < kWideMaxSlices; ++s) {
      const double f = sh.scale[s];
      const int j = b0 - sh.off[s];
      x0 += f != 0.0 && j >= 0 ? f * (double)q[s][0] : 0.0;
      x1 += f != 0.0 && j + 1 >= 0 ? f * (double)q[s][1] : 0.0;
    }
  }
  const double incl = wave_scan_dpp(x0 + x1);
  if (lane_id() == 63) sh.blk[wave_id()] = incl;
  if (t < 2) sh.b[t] = INT_MAX;
  lds_barrier();
  double base = 0.0;
  for (int q = 0; q < wave_id(); ++q) base += sh.blk[q];
  const double i1 = base + incl, i0 = i1 - x1;  // R(b0 + 1), R(b0)
  sh.pre[b0] = i0;
  sh.pre[b0 + 1] = i1;
  lds_barrier();
  WideBracket<double> o;
  o.plo = o.mlo = INFINITY;
  o.phi = o.mhi = -INFINITY;
  double slo = w.S, shi = w.S;
  if (p.min_p != 0.0) {  // kept: exp((v - M) / T) >= min_p
    const double ln = log(p.min_p);
    const double span = p.temperature * ln, e = 1e-9 * (fabs(span) + fabs(w.M)) + 1e-300;
    o.mlo = w.M + span - e;
    o.mhi = w.M + span + e;
    const double far = (w.M - o.mlo) * per + 0.01, sure = fmax((w.M - o.mhi) * per - 0.01, 0.0);
    if (far < (double)kLast) shi = fmin(shi, sh.pre[(int)far] * (1.0 + kWideRel) + kWideAbs);
    const int b = (int)fmin(sure, (double)kLast) - 2;
    slo = fmax(b >= 0 ? sh.pre[b] * (1.0 - kWideRel) - kWideAbs : 0.0, 1.0);  // the maximum's mass is 1
  }
  o.hi = o.mhi;
  if (p.top_p < 1.0) {
    const double plo = p.top_p * slo * (1.0 - kWideRel) - kWideAbs, phi = p.top_p * shi * (1.0 + kWideRel) + kWideAbs;
    // The first bin that can hold the cut, and the first whose R must have passed it.
    auto up = [&](double in) { return in * (1.0 + kWideRel) + kWideAbs >= plo; };
    auto dn = [&](double in) { return in * (1.0 - kWideRel) - kWideAbs >= phi; };
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int b = b0 + q;
      if (b > kLast) continue;
      const double in = q ? i1 : i0;
      if (up(in) && (b == 0 || !up(sh.pre[b - 1]))) atomicMin(&sh.b[0], b);
      if (dn(in) && (b == 0 || !dn(sh.pre[b - 1]))) atomicMin(&sh.b[1], b);
    }
    lds_barrier();
    const int bl = min(sh.b[0], kLast + 1), bh = sh.b[1];
    o.phi = bl == 0 ? INFINITY : w.M - ((double)bl - 0.01) / per;
    o.plo = bh == INT_MAX ? -INFINITY : w.M - ((double)bh + 2.01) / per;
    if (!(fabs(w.M) * 0x1p-48 <= 0.005 / per)) {  // a bin is no wider than the rounding of a value
      o.phi = INFINITY;
      o.plo = -INFINITY;
    }
    o.hi = fmax(o.phi, o.mhi);
  }
  return o;
}

// One workgroup per row: the row's record, and a filtered row's bracket.
template <class Src>
__global__ __launch_bounds__(kBracketThreads) void k_wide_bracket(Src src) {
  __shared__ WideBracketShared sh;
  const int64_t d = blockIdx.x;
  if (!src.takes(d)) return;
  const RowSpec r = src.spec(d);
  const WideLayout L(r.V);
  const WideKind kind = src.kind(r, L);
  if (kind != kWideWhole && kind != kWideGreedy) return;
  char* ws = src.ws(d);
  WideRow w;
  double f = 0.0, m;
  if (kind == kWideGreedy) w = wide_row_of<false>(L, ws, r, f, m);
  else w = wide_row_of<true>(L, ws, r, f, m);
  if (threadIdx.x < kWideMaxSlices) {
    const double d = (w.M - m) * wide_per_logit(r.pol);
    sh.scale[threadIdx.x] = f;
    sh.off[threadIdx.x] = d < (double)kWideBins ? (int)d : kWideBins;  // no finite token: factor 0
    L.scale(ws)[threadIdx.x] = f;
  }
  if (kind == kWideWhole && !w.bad && !wide_nofilter(r.pol)) {  // uniform
    lds_barrier();
    const WideBracket<double> B = wide_bracket(L, ws, r, w, sh);
    w.hi = B.hi;
    w.plo = B.plo;
    w.phi = B.phi;
    w.mlo = B.mlo;
    w.mhi = B.mhi;
  } else {  // every token kept (read for rows with no filter)
    w.hi = w.phi = w.mhi = -INFINITY;
    w.plo = w.mlo = INFINITY;
  }
  if (threadIdx.x == 0) {
    WideRow* o = L.row(ws);
    o->M = w.M;
    o->S = w.S;
    o->vmin = w.vmin;
    o->first = w.first;
    o->npos = w.npos;
    o->bad = w.bad;
    o->hi = w.hi;
    o->plo = w.plo;
    o->phi = w.phi;
    o->mlo = w.mlo;
    o->mhi = w.mhi;
  }
}

struct WideCollectShared {
  double rs[kWideWaves], rm[kWideWaves];
  uint32_t rn[kWideWaves], rc[kWideWaves];
  uint32_t tbits[kWideSlice / 32];
  float mv[kWideWaves][kWideSlice / kWideWaves];  // each wave's tokens whose masses are summed
};

template <class Src, int DT>
__global__ __launch_bounds__(kWideThreads) void k_wide_collect(Src src, int nS) {
  __shared__ WideCollectShared sh;
  const int t = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int64_t d = blockIdx.x / (unsigned)nS;
  const int s = (int)(blockIdx.x % (unsigned)nS);
  if (!src.takes(d)) return;
  const RowSpec r = src.spec(d);
  const WideLayout L(r.V);
  if (src.kind(r, L) != kWideWhole) return;
  char* ws = src.ws(d);
  const dsr_policy_t& p = r.pol;
  const WideRow w = *L.row(ws);
  if (w.bad) return;  // uniform
  if (wide_nofilter(p) && !wide_spread(w, p)) return;  // the records decide it
  const WideBracket<double> B{w.hi, w.plo, w.phi, w.mlo, w.mhi};
  const WideBracket<float> F = wide_bracket_f(B);
  const double M = w.M;
  const int lo = s * kWideSlice, hi = lo + kWideSlice < (int)r.V ? lo + kWideSlice : (int)r.V;
  const bool touched = wide_touched(r);
  const double* tv = L.tv<false>(ws);
  WideRec rc;
  if (touched) rc = L.rec(ws)[s];
  float v[kWidePer];
  wide_load<DT>(r, lo, t, v);
  uint32_t ok = wide_allowed<DT>(r, lo, t);
  if (touched) {
    if (t < kWideSlice / 32) sh.tbits[t] = 0u;
    lds_barrier();
    wide_touched_each<kWideThreads>(r, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi,
                                    [&](int, int32_t id) { atomicOr(&sh.tbits[(id - lo) >> 5], 1u << ((id - lo) & 31)); });
    lds_barrier();
    ok &= ~wide_bits<DT>(sh.tbits, t);
  }
  // The tokens whose masses are summed go to the wave's LDS list (they are few
  // in most rows, so their exps then fill whole waves); the listed ones are
  // only counted.  Tokens between the two cuts count for min-p alone.
  const bool mids = p.min_p != 0.0;
  float* mv = sh.mv[wave];
  uint32_t nm = 0u, sel = 0u;  // nm: uniform
#pragma unroll
  for (int k = 0; k < kWidePer; ++k) {
    const bool f = ((ok >> k) & 1u) && v[k] > -INFINITY, kp = F.kept(v[k]);
    const bool sum = f && (kp || (mids && F.middle(v[k])));
    if (f && !kp && F.listed(v[k])) sel |= 1u << k;
    const unsigned long long bal = __ballot(sum);
    if (sum) mv[nm + lanes_below(bal)] = v[k];
    nm += (uint32_t)__popcll(bal);
  }
  wave_lds_sync();
  const double iT = 1.0 / p.temperature;
  double kept = 0.0, mid = 0.0;
  uint32_t npos = 0u, nt = 0u;
  auto add = [&](double x, bool k) {
    const double e = wide_exp(wide_over(x - M, p.temperature, iT));
    kept += k ? e : 0.0;
    npos += k && e > 0.0 ? 1u : 0u;
    mid += k ? 0.0 : e;
  };
  for (uint32_t i = (uint32_t)lane; i < nm; i += 64u) add((double)mv[i], F.kept(mv[i]));
  if (touched)
    wide_touched_each<kWideThreads>(r, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi, [&](int at, int32_t) {
      const double x = tv[at];
      if (!(x > -(double)INFINITY)) return;
      const bool k = B.kept(x);
      if (k || (mids && B.middle(x))) add(x, k);
      if (!k && B.listed(x)) ++nt;
    });
  // Listed tokens go to the slice's list in thread order (a fixed order).
  const uint32_t c = (uint32_t)__popc(sel) + nt;
  const uint32_t incl = wave_scan_dpp(c);
  {
    const uint32_t np = wave_reduce_dpp(npos, OpSum());
    const double wk = wave_sum(kept), wm = wave_sum(mid);
    if (lane == 63) sh.rn[wave] = incl;
    if (lane == 0) {
      sh.rc[wave] = np;
      sh.rs[wave] = wk;
      sh.rm[wave] = wm;
    }
  }
  lds_barrier();
  uint32_t at0 = incl - c, total = 0u;
#pragma unroll
  for (int q = 0; q < kWideWaves; ++q) {
    if (q < wave) at0 += sh.rn[q];
    total += sh.rn[q];
  }
  if (total <= (uint32_t)L.cand_cap() && c) {
    double* ov = L.cand_v(ws, s);
    int32_t* oi = L.cand_i(ws, s);
#pragma unroll
    for (int k = 0; k < kWidePer; ++k)
      if ((sel >> k) & 1u) {
        ov[at0] = (double)v[k];
        oi[at0++] = (int32_t)wide_index<DT>(lo, t, k);
      }
    if (nt)
      wide_touched_each<kWideThreads>(r, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi, [&](int at, int32_t id) {
        const double x = tv[at];
        if (x > -(double)INFINITY && !B.kept(x) && B.listed(x)) {
          ov[at0] = x;
          oi[at0++] = id;
        }
      });
  }
  if (t == 0) {
    WideSum o{0.0, 0.0, 0, (int32_t)total};
    for (int q = 0; q < kWideWaves; ++q) {
      o.kept += sh.rs[q];
      o.mid += sh.rm[q];
      o.npos += (int32_t)sh.rc[q];
    }
    L.sum(ws)[s] = o;
  }
}

// ---------------------------------------------------------------------------
// Step 3.

// Tokens a finished whole row keeps, and their weights.
struct WideKeep {
  double M, T, iT, vc, min_p;
  int32_t ic;
  __device__ __forceinline__ bool in(double v, int32_t id) const { return (bool)((int)(v > vc) | ((int)(v == vc) & (int)(id <= ic))); }
  // exp((v - M) / T), or 0 below min-p.
  __device__ __forceinline__ double mass(double v) const {
    const double e = wide_exp(wide_over(v - M, T, iT));
    return e < min_p ? 0.0 : e;
  }
};

struct WideItem {  // a token of the boundary bin
  double v;
  int32_t id;
  int32_t pad;
};

struct WideCut {
  unsigned long long bm[kWideBins];  // fixed-point mass per sub-bin of the listed values
  WideItem list[kWideFine];
  double sv[kWideFine], sm[kWideFine];  // the list in rank order, and its masses
  int32_t si[kWideFine];
};

struct WideWalk {
  double vals[kWideSlice];             // the crossing slice's touched values
  uint32_t tbits[kWideSlice / 32], fbits[kWideSlice / 32];  // touched; finite ones
};

struct WideDrawShared {
  union {
    WideCut c;
    WideWalk w;
    GenShared g;   // the general path, for rows handed over
  };
  BlockScratch b;
  double Ks[kWideMaxSlices];           // kept mass per slice
  double part[2][kWideMaxSlices];
  uint32_t cnt[2][kWideMaxSlices];
  int nlist, bin, tok, margin;
  uint32_t close;
};

// Calls f(value, id) for the listed tokens of slice `wave` (lane-strided, a
// fixed order; eight loads in flight).
template <class F>
__device__ __forceinline__ void wide_listed(const WideLayout& L, char* ws, int wave, int n, F f) {
  const int w = wave < L.nS ? wave : 0;  // n is 0 past the row's slices
  const double* cv = L.cand_v(ws, w);
  const int32_t* ci = L.cand_i(ws, w);
  constexpr int U = 8;
  for (int i0 = lane_id(); i0 < n; i0 += 64 * U) {
    double v[U];
    int32_t id[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = min(i0 + 64 * u, n - 1);  // unbranched loads
      v[u] = cv[i];
      id[u] = ci[i];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + 64 * u < n) f(v[u], id[u]);
  }
}

// The min-p mass of a row (sampling.py:94-96: kept when r >= min_p * max(r)):
// the mass above the listed values and between them, and the listed tokens
// themselves.
__device__ __forceinline__ double wide_minp_mass(const WideLayout& L, char* ws, int n, const WideSum& mine, WideDrawShared& sh,
                                                 const WideKeep& K, unsigned& flags) {
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  double s = 0.0;
  uint32_t close = 0u;
  wide_listed(L, ws, wave, n, [&](double v, int32_t) {
    const double e = wide_exp(wide_over(v - K.M, K.T, K.iT));
    if (e > 0.0 && fabs(e - K.min_p) <= K.min_p * 0x1p-48) close = 1u;
    s += e < K.min_p ? 0.0 : e;
  });
  s = wave_sum(s);
  if (lane_id() == 0) sh.part[0][wave] = s + mine.kept + mine.mid;
  if (close) sh.close = 1u;
  lds_barrier();
  double S = 0.0;
  for (int q = 0; q < L.nS; ++q) S += sh.part[0][q];
  if (sh.close) flags |= DSR_FLAG_MARGIN;
  return S;
}

// The top-p cut of a whole row (sampling.py:97-102): the last kept token, by
// value and index, into K, and the kept listed mass and positive count of
// each slice into `s`, `c` of its wave.  `n` tokens are listed for this
// wave's slice; `base` is the mass certainly kept (nbase positive tokens), S
// the row's.  Returns 0 or the reason the general path must decide the row.
__device__ __forceinline__ int wide_cut(const RowSpec& r, const WideLayout& L, char* ws, const WideRow& row, int n, double base,
                                        long long nbase, double S, WideDrawShared& sh, const WideKeep& K, double& vc, int32_t& ic, double& s,
                                        uint32_t& c, unsigned& flags) {
  const int t = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int nS = L.nS;
  BlockScratch& bs = sh.b;
  // Fixed-point mass per sub-bin of the listed values, from the highest down
  // (bins of the scan's width where they have no lower end), then the sub-bin
  // that holds top_p * S.
  const double top = fmin(row.hi, row.M), low = fmin(row.plo, row.mlo);
  const double per = low > -(double)INFINITY ? 1023.0 / (top - low) : wide_per_logit(r.pol);
  auto sub = [&](double v) { return wide_bin((top - v) * per); };
  sh.c.bm[t] = 0ull;
  if (t == 0) {
    sh.bin = -1;
    sh.nlist = 0;
  }
  lds_barrier();
  wide_listed(L, ws, wave, n, [&](double v, int32_t) {
    const double e = K.mass(v);
    if (e > 0.0) atomicAdd(&sh.c.bm[sub(v)], (unsigned long long)(e * 0x1p45));
  });
  lds_barrier();
  const double P = r.pol.top_p * S;
  const long long b45 = (long long)(base * 0x1p45);
  long long tgt = (long long)(P * 0x1p45);
  if (tgt < 1) tgt = 1;
  const long long mass = (long long)sh.c.bm[t];
  long long tot;
  const long long run = b45 + block_exclusive_scan_i64(mass, bs, tot);
  if (run < tgt && tgt <= run + mass) sh.bin = t;
  lds_barrier();
  // A row that cannot be decided still takes every step below, with an empty list.
  const int bin = sh.bin;
  int why = bin < 0 ? kHandCapacity : 0;  // rounding put the boundary outside the listed tokens
  // The sub-bin's tokens, and the mass and number of listed tokens above it.
  s = 0.0;
  c = 0u;
  wide_listed(L, ws, wave, n, [&](double v, int32_t id) {
    const int b = sub(v);
    if (b < bin) {
      const double e = K.mass(v);
      s += e;
      c += e > 0.0 ? 1u : 0u;
    } else if (b == bin) {
      const int at = atomicAdd(&sh.nlist, 1);
      if (at < kWideFine) sh.c.list[at] = WideItem{v, id, 0};
    }
  });
  s = wave_sum(s);
  c = wave_reduce_dpp(c, OpSum());
  if (lane == 0) {
    sh.part[1][wave] = s;
    sh.cnt[0][wave] = c;
  }
  lds_barrier();
  int nl = sh.nlist;
  if (nl > kWideFine) why = kHandCapacity;
  if (why) nl = 0;
  double above = base;
  long long nab = nbase;
  for (int q = 0; q < nS; ++q) {
    above += sh.part[1][q];
    nab += sh.cnt[0][q];
  }
  // Rank by value, then index: the stable sort's order (:98).
  if (t < nl) {
    const WideItem me = sh.c.list[t];
    int rank = 0;
#pragma unroll 8
    for (int q = 0; q < nl; ++q) {
      const WideItem o = sh.c.list[q];
      rank += (int)(o.v > me.v) | ((int)(o.v == me.v) & (int)(o.id < me.id));
    }
    sh.c.sv[rank] = me.v;
    sh.c.sm[rank] = K.mass(me.v);
    sh.c.si[rank] = me.id;
  }
  lds_barrier();
  const double e = t < nl ? sh.c.sm[t] : 0.0;
  double ltot;
  const double before = above + block_exclusive_scan_f64(e, bs, ltot);
  const bool keep = t < nl && (before < P || (t == 0 && nab == 0));
  const int q = (int)block_sum_i64(keep ? 1 : 0, bs);
  // The last kept token starts below P and reaches it.  A bin without it: the
  // fixed-point sums (each mass cut to 2^-45) put the boundary a bin too low.
  if (!why && (q == 0 || above + ltot < P)) why = kHandCapacity;
  const double tol = ((double)(nab + q) + 16.0) * 0x1p-51 * S;
  const bool near = (t < nl && (t == q || (t == q - 1 && nab + q > 1)) && fabs(before - P) <= tol) ||
                    (t == 0 && q == nl && fabs(above + ltot - P) <= tol);
  if (block_or(near ? 1 : 0, bs)) flags |= DSR_FLAG_MARGIN;
  const double vk = sh.c.sv[q > 0 ? q - 1 : 0], vr = sh.c.sv[q < nl ? q : max(nl - 1, 0)];  // last kept, first removed
  vc = vk;
  ic = q > 0 ? sh.c.si[q - 1] : -1;
  // Values on the two sides of the cut must stay apart after (v - M) / T, or
  // the reference's probabilities could tie across it and its index order,
  // not the values', would decide.
  const double gap = 0x1p-40 * K.T;
  const bool inside = q > 0 && q < nl;
  bool apart = vk - vr >= gap;
  if (!(inside && vk != vr)) {
    double lower = -INFINITY, upper = INFINITY;
    auto side = [&](double v) {
      if (v < vr) lower = fmax(lower, v);
      if (v > vk) upper = fmin(upper, v);
    };
    wide_listed(L, ws, wave, n, [&](double v, int32_t) { side(v); });
    const double* tv = L.tv<false>(ws);
    for (int i = t; i < (int)r.pen_n; i += kThreads) side(tv[i]);
    if (t < r.prefix_n) side(tv[r.pen_n + t]);
    for (int i = t; i < (int)r.bias_n; i += kThreads) side(tv[r.pen_n + kWidePrefix + i]);
    lower = block_max(lower, bs);
    upper = -block_max(-upper, bs);
    // Untouched values are floats: a neighbour not seen here is an ulp away at least.
    const bool floats = fabs(vk) * 0x1p-25 >= gap && fabs(vr) * 0x1p-25 >= gap;
    const bool lo_ok = vr - lower >= gap, hi_ok = upper - vk >= gap;
    apart = floats && (lo_ok || !(inside || q == nl)) && (hi_ok || !(inside || q == 0));
  }
  if (!why && !apart) why = kHandOrder;
  // The bin's kept tokens, slice by slice in rank order.
  double a = 0.0;
  uint32_t ca = 0u;
  for (int i = lane; i < q; i += 64)
    if (sh.c.si[i] / kWideSlice == wave) {
      a += sh.c.sm[i];
      ca += sh.c.sm[i] > 0.0 ? 1u : 0u;
    }
  s += wave_sum(a);
  c += wave_reduce_dpp(ca, OpSum());
  return why;
}

// A whole row: the kept set (K), the kept mass per slice (sh.Ks) and in all
// (Sk), and its positive tokens.  Returns 0 or the reason the general path
// must decide the row.  Every thread of the 1,024 calls; wave w works on
// slice w.
__device__ __forceinline__ int wide_whole(const RowSpec& r, const WideLayout& L, char* ws, const WideRow& row,
                                          WideDrawShared& sh, const WideKeep& K, double& vc, int32_t& ic, double& Sk, long long& npos,
                                          unsigned& flags) {
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const dsr_policy_t& p = r.pol;
  const int nS = L.nS;
  const bool nof = wide_nofilter(p), records = nof && !wide_spread(row, p);
  WideSum mine{0.0, 0.0, 0, 0}, all{0.0, 0.0, 0, 0};
  if (!records) {
    if (lane < nS) all = L.sum(ws)[lane];
    mine.kept = lane_value(all.kept, wave);
    mine.mid = lane_value(all.mid, wave);
    mine.ncand = (int32_t)lane_value((uint32_t)all.ncand, wave);
  }
  const int n = __builtin_amdgcn_readfirstlane(mine.ncand);
  int why = __ballot(all.ncand > L.cand_cap()) ? kHandCapacity : 0;  // uniform over the workgroup
  const double base = lane_value(row_reduce(all.kept, OpSum()), 0);  // mass certainly kept, and its positive tokens
  const long long nbase = (long long)lane_value(row_reduce((uint32_t)all.npos, OpSum()), 0);
  double s = 0.0;
  uint32_t c = 0u;
  if (!nof && why == 0) {
    const double S = p.min_p != 0.0 ? wide_minp_mass(L, ws, n, mine, sh, K, flags) : row.S;
    if (p.top_p < 1.0) {
      why = wide_cut(r, L, ws, row, n, base, nbase, S, sh, K, vc, ic, s, c, flags);
    } else {  // min-p alone
      wide_listed(L, ws, wave, n, [&](double v, int32_t) {
        const double e = K.mass(v);
        s += e;
        c += e > 0.0 ? 1u : 0u;
      });
      s = wave_sum(s);
      c = wave_reduce_dpp(c, OpSum());
    }
  }
  if (lane == 0) {
    double k = 0.0;
    if (wave < nS) k = records ? L.scale(ws)[wave] * L.rec(ws)[wave].sum : mine.kept + s;
    sh.Ks[wave] = k;
    sh.cnt[1][wave] = c;
  }
  lds_barrier();
  Sk = 0.0;
  npos = records ? (long long)row.npos : nbase;
  for (int q = 0; q < nS; ++q) {
    Sk += sh.Ks[q];
    npos += sh.cnt[1][q];
  }
  return why;
}

// categorical's CDF search (sampling.py:126-128) of a whole row in index
// order: the slice whose kept mass holds u * Sk, then its tokens.
template <int DT>
__device__ __forceinline__ int64_t wide_walk(const RowSpec& r, const WideLayout& L, char* ws, WideDrawShared& sh,
                                             const WideKeep& K, double Sk, long long npos, double u, unsigned& flags) {
  const int t = threadIdx.x;
  BlockScratch& bs = sh.b;
  const double thr = u * Sk, tol = ((double)npos + 16.0) * 0x1p-51 * Sk;
  int s = -1;
  double base = 0.0, run = 0.0;
  for (int q = 0; q < L.nS; ++q) {
    const double k = sh.Ks[q];
    if (k > 0.0 && run <= thr) {
      s = q;
      base = run;
    }
    run += k;
  }
  if (s < 0) {  // not reached: Sk > 0
    flags |= DSR_FLAG_MARGIN;
    return -1;
  }
  const int64_t lo = (int64_t)s * kWideSlice, hi = lo + kWideSlice < r.V ? lo + kWideSlice : r.V;
  const bool touched = wide_touched(r);
  if (touched) {
    const WideRec rc = L.rec(ws)[s];
    const double* tv = L.tv<false>(ws);
    if (t < kWideSlice / 32) {
      sh.w.tbits[t] = 0u;
      sh.w.fbits[t] = 0u;
    }
    lds_barrier();
    // A token's value is at one place; its other places hold -inf.
    wide_touched_each<kThreads>(r, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi, [&](int at, int32_t id) {
      const double x = tv[at];
      const uint32_t bit = 1u << ((id - lo) & 31);
      atomicOr(&sh.w.tbits[(id - lo) >> 5], bit);
      if (x > -(double)INFINITY) {
        atomicOr(&sh.w.fbits[(id - lo) >> 5], bit);
        sh.w.vals[id - lo] = x;
      }
    });
    lds_barrier();
  }
  constexpr int W = 8;  // consecutive tokens per thread
  double m[W];
  double part = 0.0;
  const int64_t i0 = lo + (int64_t)t * W;
  const uint32_t aw = r.allow && i0 < hi ? (r.allow[i0 >> 5] >> (i0 & 31)) & 0xFFu : 0xFFu;
  const uint32_t tw = touched ? (sh.w.tbits[(t * W) >> 5] >> ((t * W) & 31)) & 0xFFu : 0u;
  const uint32_t fw = touched ? (sh.w.fbits[(t * W) >> 5] >> ((t * W) & 31)) & 0xFFu : 0u;
#pragma unroll
  for (int e = 0; e < W; ++e) {
    const int64_t i = i0 + e;
    double v = -INFINITY;
    if (i < hi) {
      if ((tw >> e) & 1u) v = (fw >> e) & 1u ? sh.w.vals[t * W + e] : -(double)INFINITY;
      else if ((aw >> e) & 1u)
        v = DT == DSR_BF16 ? (double)__uint_as_float((uint32_t)((const uint16_t*)r.logits)[i] << 16)
                           : (double)((const float*)r.logits)[i];
    }
    m[e] = v > -(double)INFINITY && K.in(v, (int32_t)i) ? K.mass(v) : 0.0;
    part += m[e];
  }
  double tot;
  const double at = base + block_exclusive_scan_f64(part, bs, tot);
  long long owner = block_max_i64(part > 0.0 && at <= thr ? (long long)t : -1ll, bs);
  if (owner < 0) owner = block_min_i64(part > 0.0 ? (long long)t : LLONG_MAX, bs);  // uniform
  if (owner == t) {
    double c = at;
    int64_t tok = -1;
    int margin = 1;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      if (m[e] > 0.0 && margin >= 0) {
        const double b = c;
        c += m[e];
        tok = i0 + e;
        if (c > thr) {
          margin = (c - thr <= tol || (b > 0.0 && thr - b <= tol)) ? -2 : -1;
        }
      }
    }
    sh.tok = (int)tok;
    sh.margin = margin == -1 ? 0 : 1;
  }
  __syncthreads();
  if (owner == LLONG_MAX || sh.margin) flags |= DSR_FLAG_MARGIN;
  return owner == LLONG_MAX ? -1 : (int64_t)sh.tok;
}

// A top-k row's candidates, in index order, in shu.t (cz / cid): every token
// that can survive top-k.  Returns their number, or -1 where the groups'
// 16-bit prefixes cannot bound them to the list.
template <int DT>
__device__ __forceinline__ int wide_candidates_prefix(const RowSpec& r, const WideLayout& L, char* ws, double M, long long k,
                                                      F32Shared& shu) {
  F32Lists& t = shu.t;
  BlockScratch& bs = shu.gen.b;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  uint32_t* tbm = (uint32_t*)t.sp;      // touched tokens
  uint32_t* cbm = (uint32_t*)t.pos;     // candidates
  uint16_t* base = (uint16_t*)t.kz;     // candidates below each word
  static_assert(sizeof(t.sp) >= (DSR_MAX_VOCAB + 31) / 32 * 4 && sizeof(t.pos) >= (DSR_MAX_VOCAB + 31) / 32 * 4 &&
                    sizeof(t.kz) >= 4 * kThreads * sizeof(uint16_t) && 4 * kThreads * 32 >= DSR_MAX_VOCAB,
                "bitmaps of the vocabulary");
  const int ng = L.nS * kWideGroups;  // at most 8 per thread
  uint32_t g[8];
  {
    const uint4 q = tid * 8 < ng ? *(const uint4*)(L.group(ws) + 8 * tid) : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t w4[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) g[i] = (w4[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
  }
  const uint16_t* tk = L.tk(ws);
  const double* tv = L.tv<true>(ws);
  const bool touched = wide_touched(r);
  // The thread's touched tokens, place, id and key; the first kPre history
  // entries are read once.
  constexpr int kPre = 4;
  int32_t pid[kPre];
  uint32_t pk[kPre];
#pragma unroll
  for (int i = 0; i < kPre; ++i) {
    const int e = tid + i * kThreads;
    const bool in = e < (int)r.pen_n;
    pid[i] = in ? r.pen_ids[e] : -1;
    pk[i] = in ? (uint32_t)tk[e] : 0u;
  }
  auto places = [&](auto f) {
#pragma unroll
    for (int i = 0; i < kPre; ++i)
      if (pid[i] >= 0) f(tid + i * kThreads, pid[i], pk[i]);
    for (int e = tid + kPre * kThreads; e < (int)r.pen_n; e += kThreads) f(e, r.pen_ids[e], (uint32_t)tk[e]);
    if (tid < r.prefix_n) f((int)r.pen_n + tid, r.prefix[tid], (uint32_t)tk[r.pen_n + tid]);
    for (int b = tid; b < (int)r.bias_n; b += kThreads)
      f((int)r.pen_n + kWidePrefix + b, r.bias_ids[b], (uint32_t)tk[r.pen_n + kWidePrefix + b]);
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    tbm[tid + i * kThreads] = 0u;
    cbm[tid + i * kThreads] = 0u;
  }
  if (tid == 0) t.wn[0] = 0;
  const uint32_t D = wide_floor_key(M) >> 16;
  const uint32_t tau16 = f32_tau16_each(t, wave, lane, D, k, [&](auto f) {
    for (int i = 0; i < 8; ++i) f(g[i]);
    if (touched) places([&](int, int32_t, uint32_t x) { f(x); });
  });
  if (tau16 == 0u) return -1;  // fewer finite groups and touched tokens than k
  // The groups to read again (their order does not matter), and the bitmaps.
  uint32_t* gl = &t.hist[0][0];
  constexpr int kCap = kWaves * kF32Bins;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const bool need = g[i] >= tau16;
    const unsigned long long bal = __ballot(need);
    if (bal) {  // uniform over the wave
      int at = 0;
      if (lane == 0) at = atomicAdd(&t.wn[0], (int)__popcll(bal));
      at = __builtin_amdgcn_readfirstlane(at) + (int)lanes_below(bal);
      if (need && at < kCap) gl[at] = (uint32_t)(8 * tid + i);
    }
  }
  if (touched)
    places([&](int, int32_t id, uint32_t x) {
      atomicOr(&tbm[id >> 5], 1u << (id & 31));
      if (x >= tau16) atomicOr(&cbm[id >> 5], 1u << (id & 31));
    });
  __syncthreads();
  const int n = t.wn[0];
  if (n > kCap) return -1;
  // Four lanes per group, four tokens each; two passes over the same reads
  // (the second from cache): mark the candidates, then place them.
  auto quad = [&](int item, float v[4]) -> uint32_t {  // bit e: candidate; v: values
    const int64_t i = (int64_t)gl[item >> 2] * kWideGroup + 4 * (item & 3);
    uint32_t w[4];
    wide_quad<DT>(r, i, w);
    uint32_t ok = 0xFu;
    if (i < r.V) {
      if (r.allow) ok &= r.allow[i >> 5] >> (i & 31);
      ok &= ~(tbm[i >> 5] >> (i & 31));
    }
    uint32_t sel = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = __uint_as_float(w[e]);
      if (((ok >> e) & 1u) && (f32_key(w[e], true) >> 16) >= tau16) sel |= 1u << e;
    }
    return sel;
  };
  for (int it = tid; it < 4 * n; it += kThreads) {
    float v[4];
    const uint32_t sel = quad(it, v);
    const int64_t i = (int64_t)gl[it >> 2] * kWideGroup + 4 * (it & 3);
    if (sel) atomicOr(&cbm[i >> 5], sel << (i & 31));
  }
  __syncthreads();
  // Candidates below each word: thread t owns words 4t .. 4t + 3.
  long long nc;
  {
    const uint4 q = *(const uint4*)&cbm[4 * tid];
    const uint32_t c0 = __popc(q.x), c1 = __popc(q.y), c2 = __popc(q.z), c3 = __popc(q.w);
    const long long ex = block_exclusive_scan_i64((long long)(c0 + c1 + c2 + c3), bs, nc);
    if (nc > kF32Cap) return -1;
    uint32_t b = (uint32_t)ex;
    base[4 * tid] = (uint16_t)b;
    base[4 * tid + 1] = (uint16_t)(b += c0);
    base[4 * tid + 2] = (uint16_t)(b += c1);
    base[4 * tid + 3] = (uint16_t)(b += c2);
  }
  __syncthreads();
  const double T = r.pol.temperature;
  auto place = [&](int64_t i, double v) {
    const uint32_t b = (uint32_t)(i & 31);
    const int at = (int)base[i >> 5] + __popc(cbm[i >> 5] & ((1u << b) - 1u));
    t.cz[at] = (v - M) / T;  // sampling.py:86-88, true division
    t.cid[at] = (int32_t)i;
  };
  for (int it = tid; it < 4 * n; it += kThreads) {
    float v[4];
    const uint32_t sel = quad(it, v);
    const int64_t i = (int64_t)gl[it >> 2] * kWideGroup + 4 * (it & 3);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if ((sel >> e) & 1u) place(i + e, (double)v[e]);
  }
  if (touched)
    places([&](int at, int32_t id, uint32_t x) {
      if (x >= tau16) place(id, tv[at]);
    });
  __syncthreads();
  return (int)nc;
}

// The same from the tokens themselves: the k-th largest one's whole order key,
// by four 8-bit radix passes over the row, and every token from it on.  Returns
// their number, or -1 when a tie group outgrows the list or fewer than k
// tokens are finite.  Rows that come here: many logits within 2^-7 of the k-th
// largest (nearly equal ones, or a large common offset), and a top-k near the
// row's number of 16-token groups.
template <int DT>
__device__ __forceinline__ int wide_candidates_exact(const RowSpec& r, const WideLayout& L, char* ws, double M, long long k,
                                                     F32Shared& shu) {
  F32Lists& t = shu.t;
  BlockScratch& bs = shu.gen.b;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  uint32_t* tbm = (uint32_t*)t.sp;   // touched tokens
  uint32_t* cbm = (uint32_t*)t.pos;  // candidates
  uint16_t* base = (uint16_t*)t.kz;  // candidates below each word
  const double* tv = L.tv<true>(ws);
  const bool touched = wide_touched(r);
  auto places = [&](auto f) {  // place and id
    for (int e = tid; e < (int)r.pen_n; e += kThreads) f(e, r.pen_ids[e]);
    if (tid < r.prefix_n) f((int)r.pen_n + tid, r.prefix[tid]);
    for (int b = tid; b < (int)r.bias_n; b += kThreads) f((int)r.pen_n + kWidePrefix + b, r.bias_ids[b]);
  };
  __syncthreads();  // every thread is done with the first attempt's lists
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    tbm[tid + i * kThreads] = 0u;
    cbm[tid + i * kThreads] = 0u;
  }
  __syncthreads();
  if (touched) {
    places([&](int, int32_t id) { atomicOr(&tbm[id >> 5], 1u << (id & 31)); });
    __syncthreads();
  }
  // Calls f(token, keys, bits) for each quad of untouched tokens, with every
  // thread of a wave (key 0: past the row, masked or touched).
  auto quads = [&](auto f) {
    constexpr int U = 4;
#pragma unroll 1
    for (int64_t i0 = 4 * tid; i0 - 4 * tid < r.V; i0 += 4 * kThreads * U) {
      uint32_t w[U][4], ok[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t i = i0 + 4 * kThreads * u;
        wide_quad<DT>(r, i, w[u]);
        ok[u] = i < r.V ? (r.allow ? r.allow[i >> 5] >> (i & 31) : 0xFu) : 0u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t i = i0 + 4 * kThreads * u;
        if (touched && i < r.V) ok[u] &= ~(tbm[i >> 5] >> (i & 31));
        uint32_t key[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) key[e] = f32_key(w[u][e], (ok[u] >> e) & 1u);
        f(i, key, w[u]);
      }
    }
  };
  uint32_t kth = 0u, mask = 0u;
  long long rem = k;
#pragma unroll 1
  for (int shift = 24; shift >= 0; shift -= 8) {
    *reinterpret_cast<uint4*>(&t.hist[wave][4 * lane]) = make_uint4(0u, 0u, 0u, 0u);
    wave_lds_sync();
    // A wave's keys mostly share a bin in the upper passes: the first lane's
    // bin is added once.
    auto count = [&](uint32_t key) {
      const bool on = key != 0u && (key & mask) == kth;
      const unsigned long long m = __ballot(on);
      if (m == 0ull) return;
      const uint32_t bin = (key >> shift) & 0xFFu;
      const int first = __ffsll((long long)m) - 1;
      const uint32_t b0 = lane_value(bin, first);
      const unsigned long long same = __ballot(on && bin == b0);
      if (lane == first) atomicAdd(&t.hist[wave][b0], (uint32_t)__popcll(same));
      else if (on && bin != b0) atomicAdd(&t.hist[wave][bin], 1u);
    };
    quads([&](int64_t, const uint32_t key[4], const uint32_t*) {
#pragma unroll
      for (int e = 0; e < 4; ++e) count(key[e]);
    });
    if (touched)
      places([&](int at, int32_t) {
        const double x = tv[at];
        const uint32_t key = x > -(double)INFINITY ? wide_floor_key(x) : 0u;
        if (key != 0u && (key & mask) == kth) atomicAdd(&t.hist[wave][(key >> shift) & 0xFFu], 1u);
      });
    __syncthreads();
    long long above;
    const int b = f32_pick(t, rem, above);  // uniform
    __syncthreads();
    if (b < 0) return -1;  // fewer than k finite tokens
    kth |= (uint32_t)b << shift;
    mask |= 0xFFu << shift;
    rem -= above;
  }
  // Values so close below the k-th that (v - M) / T may tie with its own
  // belong to its tie group, which the list cuts by index (sampling.py:89-91).
  {
    const double v = (double)wide_key_value(kth);
    kth = wide_floor_key(v - fabs(M - v) * 0x1p-50);
  }
  quads([&](int64_t i, const uint32_t key[4], const uint32_t*) {
    uint32_t sel = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) sel |= key[e] >= kth ? 1u << e : 0u;
    if (sel) atomicOr(&cbm[i >> 5], sel << (i & 31));
  });
  if (touched)
    places([&](int at, int32_t id) {
      const double x = tv[at];
      if (x > -(double)INFINITY && wide_floor_key(x) >= kth) atomicOr(&cbm[id >> 5], 1u << (id & 31));
    });
  __syncthreads();
  long long nc;
  {
    const uint4 q = *(const uint4*)&cbm[4 * tid];
    const uint32_t c0 = __popc(q.x), c1 = __popc(q.y), c2 = __popc(q.z), c3 = __popc(q.w);
    const long long ex = block_exclusive_scan_i64((long long)(c0 + c1 + c2 + c3), bs, nc);
    if (nc > kF32Cap) return -1;
    uint32_t b = (uint32_t)ex;
    base[4 * tid] = (uint16_t)b;
    base[4 * tid + 1] = (uint16_t)(b += c0);
    base[4 * tid + 2] = (uint16_t)(b += c1);
    base[4 * tid + 3] = (uint16_t)(b += c2);
  }
  __syncthreads();
  const double T = r.pol.temperature;
  auto place = [&](int64_t i, double v) {
    const uint32_t b = (uint32_t)(i & 31);
    const int at = (int)base[i >> 5] + __popc(cbm[i >> 5] & ((1u << b) - 1u));
    t.cz[at] = (v - M) / T;  // sampling.py:86-88, true division
    t.cid[at] = (int32_t)i;
  };
  quads([&](int64_t i, const uint32_t key[4], const uint32_t* w) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (key[e] >= kth) place(i + e, (double)__uint_as_float(w[e]));
  });
  // A token's value is at one place; its other places hold -inf.
  if (touched)
    places([&](int at, int32_t id) {
      const double x = tv[at];
      if (x > -(double)INFINITY && wide_floor_key(x) >= kth) place(id, x);
    });
  __syncthreads();
  return (int)nc;
}

// The candidates of a top-k row, or -1 with the reason.
template <int DT>
__device__ __forceinline__ int wide_candidates(const RowSpec& r, const WideLayout& L, char* ws, double M, long long k,
                                               F32Shared& shu, int& why) {
  int nc = wide_candidates_prefix<DT>(r, L, ws, M, k, shu);
  if (nc < 0) nc = wide_candidates_exact<DT>(r, L, ws, M, k, shu);  // uniform
  if (nc < 0) why = kHandCapacity;
  return nc;
}

// ---------------------------------------------------------------------------
// Step 4: the probabilities of whole rows this path decided.

template <class Src, int DT>
__global__ __launch_bounds__(kWideThreads) void k_wide_probs(Src src, int nS) {
  __shared__ uint32_t tbits[kWideSlice / 32];
  const int t = threadIdx.x;
  const int64_t d = blockIdx.x / (unsigned)nS;
  const int s = (int)(blockIdx.x % (unsigned)nS);
  if (!src.takes(d)) return;
  const RowSpec r = src.spec(d);
  const WideLayout L(r.V);
  if (src.kind(r, L) != kWideWhole) return;
  char* ws = src.ws(d);
  const WideDec dec = *L.dec(ws);
  if (dec.done != 0) return;
  const double M = L.row(ws)->M;
  const int64_t lo = (int64_t)s * kWideSlice, hi = lo + kWideSlice < r.V ? lo + kWideSlice : r.V;
  float v[kWidePer];
  wide_load<DT>(r, lo, t, v);
  uint32_t ok = wide_allowed<DT>(r, lo, t);
  const bool touched = wide_touched(r);
  WideRec rc;
  if (touched) {
    rc = L.rec(ws)[s];
    if (t < kWideSlice / 32) tbits[t] = 0u;
    __syncthreads();
    wide_touched_each<kWideThreads>(r, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi,
                                    [&](int, int32_t id) { atomicOr(&tbits[(id - lo) >> 5], 1u << ((id - lo) & 31)); });
    __syncthreads();
    ok &= ~wide_bits<DT>(tbits, t);
  }
  const WideKeep K{M, r.pol.temperature, 1.0 / r.pol.temperature, dec.vc, r.pol.min_p, dec.ic};
  auto prob = [&](double x, int32_t id) { return x > -(double)INFINITY && K.in(x, id) ? K.mass(x) / dec.Sk : 0.0; };
  constexpr int W = 4;
#pragma unroll
  for (int q = 0; q < kWidePer / W; ++q) {
    const int64_t i = wide_index<DT>(lo, t, q * W);
    double o[W];
#pragma unroll
    for (int e = 0; e < W; ++e)
      o[e] = (ok >> (q * W + e)) & 1u ? prob((double)v[q * W + e], (int32_t)(i + e)) : 0.0;
    if (r.probs_f32) {
      float* w = r.probs_f32 + i;
      if (i + W <= hi && ((uintptr_t)w & 15u) == 0) *(float4*)w = make_float4((float)o[0], (float)o[1], (float)o[2], (float)o[3]);
      else
        for (int e = 0; e < W; ++e)
          if (i + e < hi) w[e] = (float)o[e];
    }
    if (r.probs_f64) {
      double* w = r.probs_f64 + i;
      if (i + W <= hi && ((uintptr_t)w & 15u) == 0) {
        ((double2*)w)[0] = make_double2(o[0], o[1]);
        ((double2*)w)[1] = make_double2(o[2], o[3]);
      } else {
        for (int e = 0; e < W; ++e)
          if (i + e < hi) w[e] = o[e];
      }
    }
  }
  if (touched) {
    __syncthreads();  // after the zeros stored for these tokens above
    const double* tv = L.tv<false>(ws);
    wide_touched_each<kWideThreads>(r, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi, [&](int at, int32_t id) {
      const double x = tv[at];
      if (!(x > -(double)INFINITY)) return;  // masked, or counted at another place: 0
      const double o = prob(x, id);
      if (r.probs_f32) r.probs_f32[id] = (float)o;
      if (r.probs_f64) r.probs_f64[id] = o;
    });
  }
}

}  // namespace dsr
