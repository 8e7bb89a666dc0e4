// Sliced path of the speculative verifier (gfx950, wave64): requests whose
// distributions are filtered, or conditioned on a history, a bias or a mask
// (sampling.py:255-319 over :48-106).
//
// The 2K+1 distributions of every such request are rows of the sliced path
// (dsr_wide.h), with the accepted drafts before each row as its tentative
// prefix, and no probability row is written: 8 requests x 9 rows of 129,280
// would be 74 MB of float64.  What a row leaves in its workspace decides any
// token's probability:
//
//   top-k rows    their kept tokens and probabilities, in index order (at
//                 most 1,024);
//   whole rows    maximum, kept mass and last kept token: p(x) =
//                 exp((v(x) - M) / T) / S for a kept x, from x's own logit or
//                 its place among the touched values;
//   greedy rows   the first index of the maximum.
//
//   k_wide_scan, k_wide_bracket, k_wide_collect  as for sampled rows
//   k_wide_dist      one workgroup per row: the row's kept set
//   k_wide_chain     one workgroup per request: the accept chain needs 2K
//                    probabilities; a top-k request's replacement or bonus
//                    is drawn there too, from its lists
//   k_wide_residual  whole requests with a draw pending: one workgroup per
//                    8,192-token slice sums its weights
//   k_wide_resolve   the slice that holds the crossing, in index order
//
// 8 requests x 4 drafts, V = 129,280, FP32: top-k 20..200 with top-p 51.5 us
// (scan 12.6, dist 23.6, dists 4.6 with nothing to do, chain 12.6) against 730
// for a workgroup per distribution writing float64 rows and one per request
// reading them back.  The rows of the scan are read once, at the rate of a
// copy; the two single-workgroup steps are bound by their chains of
// dependent reductions and loads.
//
// A request with a row outside the path (invalid, a top-k above 1,024, a cut
// the listed values cannot decide) is built in full by k_verify_dists and
// decided by general_decide, as are float64 logits and vocabularies below
// 16,384 (8,192 where the hints say that every request is top-k or greedy).
//
// A call takes this path as a whole: one with a history, a bias or a mask, or
// one whose hints say that no request takes the fast path.  With neither, the
// requests' kinds are unknown on the host, and the launches of a second path
// would cost a batch of default policies 20 us on 63; such a call builds what
// the fast path leaves with k_verify_dists alone.
#pragma once

#include "dsr_verify.h"
#include "dsr_wide.h"

namespace dsr {

struct WideVerifyRows {
  dsr_verify_args_t v;
  VerifyLayout L;
  dsr_sample_args_t a;  // no draws; the top-k tail's status, per distribution
  __device__ __forceinline__ bool takes(int64_t) const { return true; }
  __device__ __forceinline__ WideKind kind(const RowSpec& r, const WideLayout& L) const { return wide_kind(r, L); }
  __device__ __forceinline__ char* ws(int64_t d) const { return (char*)(L.W + d * L.stride); }
  __device__ __forceinline__ RowSpec spec(int64_t d) const {
    const uint32_t row = (uint32_t)d / (uint32_t)L.slots;
    return verify_row_spec(v, L, row, (int)((uint32_t)d - row * (uint32_t)L.slots));
  }
};

// A top-k row's kept tokens, at the start of its workspace row once the row's
// records and keys have been read.
struct WideList {
  int32_t n, pad[15];
  int32_t id[kSplitMaxK];
  double p[kSplitMaxK];
};
static_assert(sizeof(WideList) <= kWideMinVocab * sizeof(double), "a workspace row holds the list");

union WideDistShared {
  F32Shared t;
  WideDrawShared w;
};

// whole: the batch may hold whole rows (their records and lists are there).
template <int DT>
__global__ __launch_bounds__(kThreads) void k_wide_dist(WideVerifyRows src, int whole) {
  __shared__ WideDistShared sh;
  const int64_t d = blockIdx.x;
  const RowSpec r = src.spec(d);
  char* ws = src.ws(d);
  const WideLayout L(r.V);
  const WideKind kind = src.kind(r, L);
  const int tid = threadIdx.x;
  int form = kFormDense, st = -1, why = 0;
  int64_t onehot = -1;
  unsigned flags = 0;
  if (kind == kWideTopK || kind == kWideGreedy) {
    double f, m;
    const WideRow w = wide_row_of<false>(L, ws, r, f, m);
    if (!w.bad && kind == kWideGreedy) {
      form = kFormOne;
      st = DSR_OK;
      onehot = w.first;
    } else if (!w.bad) {
      F32Lists& t = sh.t.t;
      const int nc = wide_candidates<DT>(r, L, ws, w.M, r.pol.top_k, sh.t, why);
      if (nc >= 0) {
        DistOut out;
        int64_t n = 0;
        st = f32_list_decide(src.a, d, r, sh.t, nc, r.pol.top_k, r.V, flags, out, n, why);
        __syncthreads();  // the list, in index order, with the tokens the filters removed at 0
        const bool few = st == kDecided;
        if (few) {
          n = nc;
          st = src.a.out_status[d];
          flags = src.a.out_flags[d];
        }
        if (st >= 0) {
          form = kFormList;
          WideList* o = (WideList*)ws;
          if (tid == 0) o->n = (int32_t)n;
          if (tid < n) {
            o->id[tid] = few ? t.cid[tid] : t.kid[tid];
            o->p[tid] = few ? t.cz[tid] : t.kz[tid];
          }
        }
      }
    }
  } else if (kind == kWideWhole && whole) {
    const WideRow w = *L.row(ws);
    if (!w.bad) {
      if (tid == 0) sh.w.close = 0u;
      lds_barrier();
      double Sk = 0.0, vc = -INFINITY;
      int32_t ic = INT32_MAX;
      long long npos = 0;
      const WideKeep every{w.M, r.pol.temperature, 1.0 / r.pol.temperature, -INFINITY, r.pol.min_p, INT32_MAX};
      why = wide_whole(r, L, ws, w, sh.w, every, vc, ic, Sk, npos, flags);
      if (why == 0) {
        form = kFormWhole;
        st = Sk > 0.0 ? DSR_OK : DSR_E_NO_MASS;
        if (tid == 0) *L.dec(ws) = WideDec{Sk, vc, ic, 0};
      }
    }
  }
  if (tid == 0) {
    int32_t* info = src.L.info + d * 4;
    info[0] = st;
    info[1] = (int32_t)onehot;
    info[2] = (int32_t)flags;
    info[3] = form;
  }
}

// A whole row's kept set as its workspace holds it, and its mass.
__device__ __forceinline__ WideKeep wide_kept(const RowSpec& r, const WideLayout& L, char* ws, double& S) {
  const WideDec c = *L.dec(ws);
  S = c.Sk;
  return WideKeep{L.row(ws)->M, r.pol.temperature, 1.0 / r.pol.temperature, c.vc, r.pol.min_p, c.ic};
}

// Token x's probability in distribution d, by one wave (every lane gets it).
__device__ __forceinline__ double wide_prob_at(const dsr_verify_args_t& a, const VerifyLayout& L, int64_t row, int slot, int32_t x) {
  const int32_t* info = L.info + (row * L.slots + slot) * 4;
  char* ws = (char*)(L.W + (row * L.slots + slot) * L.stride);
  if (info[0] != DSR_OK || x < 0 || x >= a.vocab) return 0.0;
  if (info[3] == kFormOne) return x == info[1] ? 1.0 : 0.0;
  if (info[3] == kFormList) {
    const WideList* o = (const WideList*)ws;
    const int n = o->n;
    double p = 0.0;
    for (int i = lane_id(); i < n; i += 64)
      if (o->id[i] == x) p = o->p[i];
    return wave_reduce_dpp(p, OpMax());
  }
  const RowSpec r = verify_row_spec(a, L, row, slot);
  const WideLayout W(r.V);
  double S;
  const WideKeep k = wide_kept(r, W, ws, S);
  // Its place among the touched values: the history's, the prefix's first, the bias's.
  int64_t at = -1;
  int e0 = 0, e1 = 0;
  if (r.pen_n > 0) wide_range(r.pen_ids, (int)r.pen_n, x, x + 1, e0, e1);
  if (e1 > e0) at = e0;
  for (int q = 0; q < r.prefix_n && at < 0; ++q)
    if (r.prefix[q] == x) at = r.pen_n + q;
  if (at < 0 && r.bias_n > 0) {
    wide_range(r.bias_ids, (int)r.bias_n, x, x + 1, e0, e1);
    if (e1 > e0) at = r.pen_n + kWidePrefix + e0;
  }
  double v = -INFINITY;
  if (at >= 0) v = W.tv<false>(ws)[at];
  else if (allowed_bit(r.allow, x)) v = load_logit(r.logits, r.dtype, x);
  return v > -(double)INFINITY && k.in(v, x) ? k.mass(v) / S : 0.0;
}

// The draw over a top-k request's lists: max(p - q, 0) in index order
// (sampling.py:131-139, then :118-128), a kept token per thread.
__device__ __forceinline__ int wide_list_draw(const WideList* P, const WideList* Q, double u, int32_t* qid, double* qp,
                                              BlockScratch& bs, int32_t* tok, int64_t& rep, int& used, unsigned& flags) {
  const int t = threadIdx.x;
  const int n = P->n, m = Q ? Q->n : 0;
  if (t < m) {
    qid[t] = Q->id[t];
    qp[t] = Q->p[t];
  }
  const int32_t id = t < n ? P->id[t] : INT32_MAX;
  double x = t < n ? P->p[t] : 0.0;
  __syncthreads();
  int lo = 0, hi = m;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (qid[mid] < id) lo = mid + 1; else hi = mid;
  }
  if (lo < m && qid[lo] == id) x = fmax(x - qp[lo], 0.0);
  double total;
  const double before = block_exclusive_scan_f64(x, bs, total);
  const long long npos = block_sum_i64(x > 0.0 ? 1 : 0, bs);
  used = 0;
  if (Q && (!(total > 0.0) || !isfinite(total))) return DSR_E_CORRECTION;
  long long pick;
  if (npos == 1) {  // a single positive token: no uniform is drawn (sampling.py:120-122)
    pick = block_max_i64(x > 0.0 ? (long long)t : -1ll, bs);
  } else {
    if (!(u >= 0.0 && u < 1.0)) return DSR_E_UNIFORM;
    used = 1;
    const double thr = u * total, tol = ((double)npos + 16.0) * 0x1p-51 * total + 0x1p-46;
    pick = block_min_i64(x > 0.0 && before + x > thr ? (long long)t : LLONG_MAX, bs);
    bool margin = pick == LLONG_MAX;  // rounding left no crossing: the last positive token
    if (margin) pick = block_max_i64(x > 0.0 ? (long long)t : -1ll, bs);
    margin = margin || (pick == t && (before + x - thr <= tol || (before > 0.0 && thr - before <= tol)));
    if (block_or(margin ? 1 : 0, bs)) flags |= DSR_FLAG_MARGIN;
  }
  if (pick == t) *tok = id;
  __syncthreads();
  rep = *tok;
  return DSR_OK;
}

// The weights of a whole request's draw: p_j (bonus), or max(p_j - q_j, 0).
// Both rows have the same touched places and mask.
struct WideWeights {
  RowSpec p, q;
  char *wp, *wq;
  WideKeep kp, kq;
  double sp, sq;
  bool resid;
  __device__ __forceinline__ double operator()(double vp, double vq, int32_t id) const {
    const double x = vp > -(double)INFINITY && kp.in(vp, id) ? kp.mass(vp) / sp : 0.0;
    if (!resid) return x;
    const double y = vq > -(double)INFINITY && kq.in(vq, id) ? kq.mass(vq) / sq : 0.0;
    return fmax(x - y, 0.0);
  }
};

// Whether request `row` draws here; sets its weights.
__device__ __forceinline__ bool wide_pending(const dsr_verify_args_t& a, const VerifyLayout& L, int64_t row, WideWeights& w) {
  const int64_t d0 = row * L.slots;
  if (!wide_request(L, row) || L.info[d0 * 4 + 3] != kFormWhole) return false;
  const Decision& d = L.dec[row];
  if (d.status != DSR_OK || d.next == 0) return false;
  const WideLayout W(a.vocab);
  const int j = d.draw_j;
  w.resid = d.next == 1;
  w.p = verify_row_spec(a, L, row, j);
  w.wp = (char*)(L.W + (d0 + j) * L.stride);
  w.kp = wide_kept(w.p, W, w.wp, w.sp);
  w.q = w.p;
  w.wq = w.wp;
  w.kq = w.kp;
  w.sq = w.sp;
  if (w.resid) {
    w.q = verify_row_spec(a, L, row, a.K + 1 + j);
    w.wq = (char*)(L.W + (d0 + a.K + 1 + j) * L.stride);
    w.kq = wide_kept(w.q, W, w.wq, w.sq);
  }
  return true;
}

struct WideResidualShared {
  double s[kWideWaves];
  uint32_t n[kWideWaves], f[kWideWaves];
  uint32_t tbits[kWideSlice / 32];
};

template <int DT>
__global__ __launch_bounds__(kWideThreads) void k_wide_residual(dsr_verify_args_t a, VerifyLayout L, int nS) {
  __shared__ WideResidualShared sh;
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x / (unsigned)nS;
  const int s = (int)(blockIdx.x % (unsigned)nS);
  WideWeights w;
  if (!wide_pending(a, L, row, w)) return;
  const WideLayout W(a.vocab);
  const int lo = s * kWideSlice, hi = lo + kWideSlice < (int)a.vocab ? lo + kWideSlice : (int)a.vocab;
  float vp[kWidePer], vq[kWidePer];
  wide_load<DT>(w.p, lo, t, vp);
  wide_load<DT>(w.q, lo, t, vq);
  uint32_t ok = wide_allowed<DT>(w.p, lo, t);
  const bool touched = wide_touched(w.p);
  WideRec rc;
  if (touched) {
    rc = W.rec(w.wp)[s];
    sh.tbits[t] = 0u;
    lds_barrier();
    wide_touched_each<kWideThreads>(w.p, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi,
                                    [&](int, int32_t id) { atomicOr(&sh.tbits[(id - lo) >> 5], 1u << ((id - lo) & 31)); });
    lds_barrier();
    ok &= ~wide_bits<DT>(sh.tbits, t);
  }
  double sum = 0.0;
  uint32_t npos = 0u, first = (uint32_t)INT32_MAX;
  auto add = [&](double x, double y, int32_t id) {
    const double m = w(x, y, id);
    sum += m;
    if (m > 0.0) {
      ++npos;
      first = min(first, (uint32_t)id);
    }
  };
  // Tokens the target row cut weigh nothing: a wave without any skips the exps.
#pragma unroll
  for (int k = 0; k < kWidePer; ++k) {
    const int32_t id = (int32_t)wide_index<DT>(lo, t, k);
    const bool in = ((ok >> k) & 1u) && vp[k] > -INFINITY && w.kp.in((double)vp[k], id);
    if (__ballot(in))
      if (in) add((double)vp[k], (double)vq[k], id);
  }
  if (touched) {
    const double *tp = W.tv<false>(w.wp), *tq = W.tv<false>(w.wq);
    wide_touched_each<kWideThreads>(w.p, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi, [&](int at, int32_t id) { add(tp[at], tq[at], id); });
  }
  sum = wave_sum(sum);
  npos = wave_reduce_dpp(npos, OpSum());
  first = wave_reduce_dpp(first, OpMin());
  if (lane_id() == 0) {
    sh.s[wave_id()] = sum;
    sh.n[wave_id()] = npos;
    sh.f[wave_id()] = first;
  }
  lds_barrier();
  if (t == 0) {
    DrawPart o{0.0, 0, INT32_MAX, 0};
    for (int q = 0; q < kWideWaves; ++q) {
      o.sum += sh.s[q];
      o.npos += sh.n[q];
      o.first = min(o.first, (long long)sh.f[q]);
    }
    L.dpart[row * kDrawSplit + s] = o;
  }
}
static_assert(kWideMaxSlices <= kDrawSplit && kWideSlice / 32 == kWideThreads, "a part per slice, a word per thread");

struct WideResolveShared {
  BlockScratch b;
  double vals[kWideSlice];                                   // the slice's touched weights
  uint32_t tbits[kWideSlice / 32], fbits[kWideSlice / 32];  // touched; positive ones
  int tok, margin;
};

template <int DT>
__global__ __launch_bounds__(kThreads) void k_wide_resolve(dsr_verify_args_t a, VerifyLayout L) {
  __shared__ WideResolveShared sh;
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x;
  WideWeights w;
  if (!wide_pending(a, L, row, w)) return;
  const WideLayout W(a.vocab);
  Decision d = L.dec[row];
  // Every thread reads the slices' parts: sums in slice order.
  const DrawPart* parts = L.dpart + row * kDrawSplit;
  double total = 0.0;
  long long npos = 0, first = INT32_MAX;
  for (int q = 0; q < W.nS; ++q) {
    total += parts[q].sum;
    npos += parts[q].npos;
    first = min(first, parts[q].first);
  }
  int64_t rep = -1;
  int used = 0, st = DSR_OK;
  double u = 0.0;
  if (w.resid && (!(total > 0.0) || !isfinite(total))) {
    st = DSR_E_CORRECTION;
  } else if (npos == 1) {
    rep = first;  // a single positive token: no uniform is drawn (sampling.py:120-122)
  } else {
    if (a.rng_target) pcg64_draws(a.rng_target + 4 * row, 1, &u);
    else u = a.u_target[row];
    if (!(u >= 0.0 && u < 1.0)) st = DSR_E_UNIFORM;
    else used = 1;
  }
  if (used) {  // uniform
    // The last slice with mass that starts at or below the crossing.
    const double thr = u * total, tol = ((double)npos + 16.0) * 0x1p-51 * total + 0x1p-46;
    int s = 0;
    double base = 0.0, run = 0.0;
    for (int q = 0; q < W.nS; ++q) {
      const double k = parts[q].sum;
      if (k > 0.0 && run <= thr) {
        s = q;
        base = run;
      }
      run += k;
    }
    const int lo = s * kWideSlice, hi = lo + kWideSlice < (int)a.vocab ? lo + kWideSlice : (int)a.vocab;
    const bool touched = wide_touched(w.p);
    if (t < kWideSlice / 32) {
      sh.tbits[t] = 0u;
      sh.fbits[t] = 0u;
    }
    lds_barrier();  // the clear bitmaps
    if (touched) {
      const WideRec rc = W.rec(w.wp)[s];
      const double *tp = W.tv<false>(w.wp), *tq = W.tv<false>(w.wq);
      wide_touched_each<kThreads>(w.p, rc.e0, rc.e1, rc.b0, rc.b1, lo, hi, [&](int at, int32_t id) {
        const double x = w(tp[at], tq[at], id);
        const uint32_t bit = 1u << ((id - lo) & 31);
        atomicOr(&sh.tbits[(id - lo) >> 5], bit);
        if (x > 0.0) {  // a token's value is at one place; its other places hold -inf
          atomicOr(&sh.fbits[(id - lo) >> 5], bit);
          sh.vals[id - lo] = x;
        }
      });
      lds_barrier();
    }
    constexpr int N = kWideSlice / kThreads;  // consecutive tokens per thread
    static_assert(N == 8, "a byte of each bitmap per thread");
    const int i0 = lo + t * N;
    const uint32_t aw = w.p.allow && i0 < hi ? (w.p.allow[i0 >> 5] >> (i0 & 31)) & 0xFFu : 0xFFu;
    const uint32_t tw = (sh.tbits[t >> 2] >> (8 * (t & 3))) & 0xFFu, fw = (sh.fbits[t >> 2] >> (8 * (t & 3))) & 0xFFu;
    double m[N], part = 0.0;
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const int i = min(i0 + e, hi - 1);  // unbranched loads
      const double x = logit_as<DT>((const char*)w.p.logits, i), y = w.resid ? (double)logit_as<DT>((const char*)w.q.logits, i) : -(double)INFINITY;
      m[e] = 0.0;
      if (i0 + e < hi) {
        if ((tw >> e) & 1u) m[e] = (fw >> e) & 1u ? sh.vals[t * N + e] : 0.0;
        else if ((aw >> e) & 1u) m[e] = w(x, y, i);
      }
      part += m[e];
    }
    double tot;
    const double at = base + block_exclusive_scan_f64(part, sh.b, tot);
    long long owner = block_max_i64(part > 0.0 && at <= thr ? (long long)t : -1ll, sh.b);
    if (owner < 0) owner = block_min_i64(part > 0.0 ? (long long)t : LLONG_MAX, sh.b);
    if (owner == t) {
      double c = at;
      int tok = -1, margin = 1;
      bool found = false;
#pragma unroll
      for (int e = 0; e < N; ++e) {
        if (m[e] > 0.0 && !found) {
          const double b = c;
          c += m[e];
          tok = i0 + e;
          if (c > thr) {
            found = true;
            margin = (c - thr <= tol || (b > 0.0 && thr - b <= tol)) ? 1 : 0;
          }
        }
      }
      sh.tok = tok;
      sh.margin = margin;
    }
    __syncthreads();
    rep = sh.tok;  // the slice has mass: one thread owned it
    if (sh.margin) d.flags |= DSR_FLAG_MARGIN;
  }
  if (t == 0) {
    if (st != DSR_OK) {
      d.status = st;
    } else {
      const Request rq = request_of(a, row);
      verify_append(a, rq, d, rep, used);
    }
    write_decision(a, row, d);
  }
}

struct WideChainShared {
  double prob[2 * DSR_MAX_DRAFTS + 1];
  double qp[kSplitMaxK];
  int32_t qid[kSplitMaxK];
  int32_t tok;
};
static_assert(2 * DSR_MAX_DRAFTS + 1 <= kWaves, "a wave per distribution");

// Request `row` of the sliced path: the accept chain, and a greedy or top-k
// request's last token.  A whole request's draw is left to k_wide_residual
// and k_wide_resolve.
__device__ __forceinline__ void wide_decide(const dsr_verify_args_t& a, const VerifyLayout& L, int64_t row, WideChainShared& ws,
                                            BlockScratch& bs, Decision& d, double* ua) {
  const int K = a.K;
  const int32_t* info = L.info + row * L.slots * 4;
  const bool greedy = a.policy[row].temperature == 0.0;
  const int slot = __builtin_amdgcn_readfirstlane(wave_id());
  if (slot < (int)L.slots && slot != K) {
    const int j = slot < K ? slot : slot - K - 1;
    const double p = wide_prob_at(a, L, row, slot, a.draft_ids[row * K + j]);
    if (lane_id() == 0) ws.prob[slot] = p;
  }
  __syncthreads();
  Request rq = request_of(a, row);
  if (a.rng_accept) rq.ua = ua;  // the accept domain's next K draws, consumed in order
  if (threadIdx.x == 0) {
    auto status_of = [&](int s) { return (int)info[s * 4]; };
    if (a.rng_accept) pcg64_draws(a.rng_accept + 4 * row, K, ua);
    verify_precheck(a, rq, status_of, d);
    for (int j = 0; j < K; ++j) d.flags |= (unsigned)info[(K + 1 + j) * 4 + 2] & DSR_FLAG_MARGIN;
    // p and q each carry the rounding of their sum, below 2^-46 relative.
    if (d.status == DSR_OK)
      verify_chain(
          a, rq, greedy, 0x1p-45, status_of, [&](int s, int) { return ws.prob[s]; },
          [&](int j) { return (int64_t)info[j * 4 + 1]; },
          [&](int j) { d.flags |= (unsigned)info[j * 4 + 2] & DSR_FLAG_MARGIN; }, d);
  }
  __syncthreads();
  if (d.status == DSR_OK && d.next != 0) {
    const int j = d.draw_j;
    if (!greedy && info[3] == kFormWhole) {
      if (threadIdx.x == 0) L.dec[row] = d;
      return;
    }
    int64_t rep = info[j * 4 + 1];
    int used = 0, st = DSR_OK;
    unsigned flags = 0;
    if (!greedy) {
      double u = 0.0;
      if (a.rng_target) pcg64_draws(a.rng_target + 4 * row, 1, &u);
      else u = a.u_target[row];
      auto list = [&](int s) { return (const WideList*)(L.W + (row * L.slots + s) * L.stride); };
      st = wide_list_draw(list(j), d.next == 1 ? list(K + 1 + j) : nullptr, u, ws.qid, ws.qp, bs, &ws.tok, rep, used, flags);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      d.flags |= flags;
      if (st != DSR_OK) d.status = st; else verify_append(a, rq, d, rep, used);
    }
  }
  if (threadIdx.x == 0) {
    L.dec[row] = d;
    L.dec[row].next = 0;  // nothing is pending
    write_decision(a, row, d);
  }
}

__global__ __launch_bounds__(kThreads) void k_wide_chain(dsr_verify_args_t a, VerifyLayout L) {
  __shared__ union {
    WideChainShared w;
    GenShared g;
  } sh;
  __shared__ BlockScratch bs;
  __shared__ Decision d;
  __shared__ double ua[DSR_MAX_DRAFTS];
  const int64_t row = blockIdx.x;
  if (wide_request(L, row)) wide_decide(a, L, row, sh.w, bs, d, ua);
  else general_decide(a, L, row, sh.g, d);
}

}  // namespace dsr
