/* The wide nucleus path: ids only, k > 4096 on rows longer than the nucleus
 * kernel takes (top-k disabled on a text vocabulary), gfx950 wave64.  The op
 * graph's definition (src/sampling.c:22-49), bit for bit, without a sort.
 *
 * The id is the first maximum of p_r / -log(1 - u_r) over the kept ranks, so it
 * takes the exact cut, the exact kept sum and the elements of the few ranks
 * that can win.  k_sel_max and k_sel_hist (d3s_select.hip) first count and sum
 * each row's elements by bucket below its max; then
 *  k_nuc_bound (a workgroup per row): each bucket's first rank, and the buckets
 *     that can hold the cut, from the exact sums' bounds;
 *  k_nuc_race (a workgroup per share of the ranks): each rank's e = exp(x - m)
 *     being known to 1/SEL_SCALE from its bucket, the ranks whose score can reach
 *     the best score some surely kept rank of the share has (one or two);
 *  k_nuc_gather (a workgroup per segment): the elements of the cut's buckets and
 *     of the buckets of those ranks that can reach the row's best, and the exact
 *     sum of fix40(d3s_expf(x - lse)) before the cut's;
 *  k_nuc_final (a workgroup per row): the cut and the kept sum exactly, the
 *     ranks' elements (by sorting a small gathered set, by counting 11 bits of
 *     what its keys span in a large one: crowded ties, top_p near 1), their exact
 *     scores and the id.
 * A row no rank of which can score (u = 0 throughout) is its first rank's.  One
 * whose kept ranks alone have no positive score, or with more candidates than
 * k_nuc_race files, is sorted by k_nuc_final's workgroup (1.4 ms at V = 151 936).
 *
 * Bound: k_sel_hist's exponentials and each launch's latency.  [64, 151936]
 * bf16, N(0, 3) logits, top_p 0.9: 4.3 + 15.9 + 9.0 + 8.9 + 12.9 + 11.8 us (60 us
 * a call) against 167 us for the sorting kernels, and at any T (T = 1e-5: 48
 * against 241 us); top_p 1: 148 against 174 us; N(0, 0.3) logits (93% of the ranks
 * kept) 140 against 174 us; one row 42 against 68 us, 72 against 75 us at top_p 1.
 * Not everywhere: [64, 151936] of whole numbers at top_p 1 202 against 167 us, of
 * one value 153 against 118 us (thousands of equal elements at the cut, searched
 * by one workgroup a row). */
#include <algorithm>

#include "d3s_select.h"

#pragma clang fp contract(off)

namespace d3s {

constexpr int NU_C = 32; /* candidate ranks a share files */

struct NucRow {
  float M, lse;
  uint32_t state;  /* NucState */
  uint32_t b1, b2; /* the buckets the cut lies in; b1 > b2: the cut is k */
  uint32_t n1;     /* the elements before b1, and (q1) their sum of fix40(d3s_expf(x - m)) */
  uint32_t r1, r2; /* the ranks below r1 are kept, those from r2 on are not */
  uint32_t open;   /* the cut is k unless it lies in b1 .. b2 (nothing, or nothing of any mass, follows) */
  uint64_t q1, qk; /* qk: the sum of all k (b1 > b2, or open) */
};
/* a share of the ranks: the least its best kept rank can score, and the ranks
 * that can score as much, with the most they can, their buckets and the
 * buckets' first ranks */
struct NucShare {
  float best;
  uint32_t n;
  uint32_t rank[NU_C], bucket[NU_C], start[NU_C];
  float most[NU_C];
};
struct NucSeg {
  uint32_t na, nb; /* elements gathered: of the cut's buckets, of the candidates' other buckets */
  uint64_t psum;   /* sum of fix40(d3s_expf(x - lse)) before the cut's buckets */
};
struct NucLayout {
  uint64_t *keys;  /* [n][2][vstride]: the two gathered sets, segment s's at s rstride */
  uint32_t *start; /* [n][SEL_NB]: each bucket's first rank */
  NucRow *row;     /* [n] */
  NucSeg *seg;     /* [n][BK_SMAX] */
  NucShare *share; /* [n][BK_SMAX] */
  int64_t vstride;
  int rstride, nseg;
};

namespace {

enum NucState : uint32_t { NUC_LIVE, NUC_REFUSED, NUC_MASKED };
constexpr int NU_T = 1024, NU_NW = NU_T / WAVE;
constexpr uint32_t NU_SMALL = 512; /* gathered elements ranked by counting (a pass over all for each; past
                                      that a search narrows them, about three passes) */
constexpr int NR_T = 512;          /* threads of a share's workgroup */
constexpr uint32_t NU_TOP = 512;   /* every share first looks at the first ranks */

/* exclusive block scan of per-thread 64-bit values modulo 2^64; tot = total.
 * Ends with a barrier. */
__device__ __forceinline__ uint64_t nuc_scan(uint64_t v, uint64_t *sh, uint64_t &tot) {
  const int lane = lane_id(), wid = (int)threadIdx.x / WAVE;
  const uint64_t inc = wave_scan_mod64(v);
  if (lane == WAVE - 1) sh[wid] = inc;
  __syncthreads();
  uint64_t base = 0ull, t = 0ull;
#pragma unroll
  for (int w = 0; w < NU_NW; w++) {
    const uint64_t x = sh[w];
    base += w < wid ? x : 0ull;
    t += x;
  }
  __syncthreads();
  tot = t;
  return base + inc - v;
}

/* the same for a count as well (shn: NU_NW words) */
__device__ __forceinline__ uint64_t nuc_scan2(uint64_t v, uint32_t c, uint64_t *sh, uint32_t *shn, uint64_t &tot,
                                              uint32_t &before, uint32_t &n) {
  const int lane = lane_id(), wid = (int)threadIdx.x / WAVE;
  const uint64_t inc = wave_scan_mod64(v);
  const uint32_t cin = wave_scan_add_u32(c);
  if (lane == WAVE - 1) {
    sh[wid] = inc;
    shn[wid] = cin;
  }
  __syncthreads();
  uint64_t base = 0ull, t = 0ull;
  uint32_t cb = 0u, ct = 0u;
#pragma unroll 4
  for (int w = 0; w < NU_NW; w++) {
    const uint64_t x = sh[w];
    const uint32_t y = shn[w];
    base += w < wid ? x : 0ull;
    cb += w < wid ? y : 0u;
    t += x;
    ct += y;
  }
  __syncthreads();
  tot = t;
  before = cb + cin - c;
  n = ct;
  return base + inc - v;
}

/* bounds of exp(z) over bucket b (a margin of 2^-14 covers z's rounding, the
 * bucket's edges and v_exp_f32) */
__device__ __forceinline__ float nuc_ehi(int b) {
  return __builtin_amdgcn_exp2f((float)b * (-LOG2E_F / SEL_SCALE)) * (1.0f + 0x1p-14f);
}
__device__ __forceinline__ float nuc_elo(int b) {
  return b >= SEL_NB - 1 ? 0.0f : __builtin_amdgcn_exp2f((float)(b + 1) * (-LOG2E_F / SEL_SCALE)) * (1.0f - 0x1p-14f);
}

/* whether a kept rank's score p / -log(1 - u) can be positive: 1 - u, as
 * rounded, in (0, 1) (at 1 the noise is -0 and the score -inf; at 0 it is 0) */
__device__ __forceinline__ bool nuc_races(float u) {
  const float w = 1.0f - u;
  return w < 1.0f && w > 0.0f;
}

/* bounds of the race's noise -d3s_logf(1 - u) for those u: from 2^-8 on the
 * hardware log (its error, at most 2^-23 |log2| + 2^-24, and 1 - u's rounding
 * are below 2^-14 of it there); below, u <= -log(1 - u) <= u + u^2, within
 * 2^-24 for 1 - u's rounding and the log's, and at least 2^-24 (1 - u, as
 * rounded, is at most 1 - 2^-24; the log's relative error there is 2^-24): without
 * that a rank with u = 2^-24, one in 2^24, would count as able to win from
 * anywhere, and the bucket of a row's far tail be gathered and searched */
constexpr float NU_LEAST = 0x1p-24f * (1.0f - 0x1p-12f);
__device__ __forceinline__ float nuc_noise_hi(float u) {
  const float a = -__builtin_amdgcn_logf(1.0f - u) * (LN2_F * (1.0f + 0x1p-12f));
  const float b = (__builtin_fmaf(u, u, u) + 0x1p-24f) * (1.0f + 0x1p-16f);
  return u < 0x1p-8f ? b : a;
}
__device__ __forceinline__ float nuc_noise_lo(float u) {
  const float a = -__builtin_amdgcn_logf(1.0f - u) * (LN2_F * (1.0f - 0x1p-12f));
  const float b = fmaxf((u - 0x1p-24f) * (1.0f - 0x1p-16f), NU_LEAST);
  return u < 0x1p-8f ? b : a;
}

/* the bucket of rank r (start: SEL_NB + 1 entries, start[SEL_NB] > r) */
__device__ __forceinline__ int nuc_bucket_of(const uint32_t *start, uint32_t r) {
  int b = 0;
#pragma unroll
  for (int step = SEL_NB / 2; step >= 1; step >>= 1) b += start[b + step] <= r ? step : 0;
  return b;
}

__global__ __launch_bounds__(NU_T) void k_nuc_bound(SampleArgs a, SelLayout F, NucLayout N) {
  __shared__ uint32_t start[SEL_NB + 1];
  __shared__ uint32_t sh[NU_NW];
  __shared__ uint64_t sq[NU_NW], qv[3];
  __shared__ int first_cut, all_drop, kth;
  const int row = (int)blockIdx.x, tid = (int)threadIdx.x;
  /* this thread's two buckets over the segments */
  uint2 cs[BK_SMAX];
  ulonglong2 qs[BK_SMAX];
  const size_t at = (size_t)row * F.nseg * SEL_NB + 2 * tid;
#pragma unroll
  for (int s = 0; s < BK_SMAX; s++)
    if (s < F.nseg) {
      cs[s] = *(const uint2 *)(F.cnt + at + (size_t)s * SEL_NB);
      qs[s] = *(const ulonglong2 *)(F.csum + at + (size_t)s * SEL_NB);
    }
  const RowP rp = row_params(a, row);
  const float T = rp.T, top_p = rp.top_p;
  NucRow *out = N.row + row;
  float M;
  const SelRow what = sel_row_max(F, row, T, M);
  if (what != SEL_LIVE) {
    if (tid == 0) out->state = what == SEL_MASKED ? NUC_MASKED : NUC_REFUSED;
    return;
  }
  uint32_t c[2] = {0u, 0u};
  uint64_t q[2] = {0ull, 0ull};
#pragma unroll
  for (int s = 0; s < BK_SMAX; s++)
    if (s < F.nseg) {
      c[0] += cs[s].x;
      c[1] += cs[s].y;
      q[0] += qs[s].x;
      q[1] += qs[s].y;
    }
  if (tid == 0) first_cut = all_drop = kth = SEL_NB;
  uint32_t n_all;
  uint64_t S;
  const uint32_t r0 = block_excl_scan_u32<NU_NW>(c[0] + c[1], sh, n_all);
  const uint64_t p0 = nuc_scan(q[0] + q[1], sq, S);
  /* (the last bucket's count is what the others leave of the row) */
  if (tid == NU_T - 1) c[1] = (uint32_t)a.vocab - n_all;
  start[2 * tid] = r0;
  start[2 * tid + 1] = r0 + c[0];
  ((uint2 *)(N.start + (size_t)row * SEL_NB))[tid] = make_uint2(r0, r0 + c[0]);
  if (tid == 0) start[SEL_NB] = (uint32_t)a.vocab;
  const float lse = M + d3s_logf(d3s_fixsum_to_f32(S));
  const uint32_t k = (uint32_t)a.k;

  /* c_r = RN(P_r 2^-40), P_r the sum of fix40(d3s_expf(x_j - lse)) over j <= r,
   * against Q_r, the sum of fix40(d3s_expf(x_j - m)): each term of either is short
   * of its real value by less than a unit, and exp(x_j - lse) is exp(x_j - m) g,
   * g = exp(-(lse - m)), whatever lse's own rounding (the largest part of x_j - lse
   * for a large |lse|: T near 0).  What is left are the roundings of x_j - lse
   * (2^-24 of at most 28: a term further down is zero), of x_j - m (28 + lse - m)
   * and of lse - m, and three d3s_expf's (2^-23 each, counted twice), in all
   * (68 + 2 (lse - m)) 2^-24.  So
   *   Q g (1 - eps) - (r + 1) <= P_r <= (Q + r + 1) g (1 + eps). */
  const float over = lse - M;
  const double tq = (double)top_p * 0x1p40, g = (double)d3s_expf(-over);
  const double eps = (double)(76.0f + 2.125f * over) * 0x1p-24;
  const double g_hi = g * (1.0 + eps) * (1.0 + 0x1p-22), g_lo = g * (1.0 - eps);
  /* the last bucket with a term of P that is not zero (x - lse > -27.73) */
  const int bz = (int)fminf(fmaxf((27.75f - over) * SEL_SCALE + 2.0f, 0.0f), (float)(SEL_NB - 1));
  {
    uint32_t n = r0;
    uint64_t Q = p0;
    int vs = SEL_NB, va = SEL_NB, vk = SEL_NB;
#pragma unroll
    for (int e = 0; e < 2; e++) {
      n += c[e];
      Q += q[e];
      if (c[e]) {
        const double nd = 1.001 * (double)n;
        const bool some = ((double)Q + nd) * g_hi > tq;
        const bool all = (double)Q * g_lo - nd - 2.0 > tq + fabs(tq) * 0x1p-22;
        if (some) vs = min(vs, 2 * tid + e); /* its last rank may be dropped */
        if (all) va = min(va, 2 * tid + e);  /* its last rank certainly is */
        if (n >= k) vk = min(vk, 2 * tid + e);
      }
    }
    vs = wave_min_i32(vs); /* (an atomic a wave, not one a bucket past the cut) */
    va = wave_min_i32(va);
    vk = wave_min_i32(vk);
    if (lane_id() == 0) {
      atomicMin(&first_cut, vs);
      atomicMin(&all_drop, va);
      atomicMin(&kth, vk);
    }
  }
  __syncthreads();
  const int bk = kth;
  if (tid == bk / 2) {
    qv[1] = p0 + q[0] + (bk & 1 ? q[1] : 0ull);
    qv[2] = q[bk & 1];
  }
  const int fc = first_cut;
  const bool none = fc > bk || fc > bz; /* no rank below k is dropped */
  const int b1 = none ? bk : fc, b2 = none ? bk : min(all_drop, bk);
  if (tid == b1 / 2) qv[0] = p0 + (b1 & 1 ? q[0] : 0ull);
  __syncthreads();
  /* all k's sum is known when they end with a bucket, or in one of zero terms;
   * then only the buckets that can hold the cut are looked at */
  const bool known = start[bk + 1] == k || qv[2] == 0ull;
  const bool whole = none && known, open = !none && known && b2 == bk;
  /* R1 ranks are surely kept (rank 0 always is), none past R2 is */
  uint32_t R1 = k;
  const uint32_t R2 = none ? k : min(k, start[b2 + 1]);
  if (!none) {
    const double step = (double)nuc_ehi(b1) * 0x1p40 + 1.0;
    double j = (tq / g_hi - (double)qv[0] - 1.001 * (double)start[b1]) / step - 2.0;
    j = j > 0.0 ? j : 0.0;
    const double most = (double)(start[b1 + 1] - start[b1]);
    R1 = start[b1] + (uint32_t)(j < most ? j : most);
    R1 = min(max(R1, 1u), R2);
  }

  if (tid == 0) {
    NucRow r;
    r.M = M;
    r.lse = lse;
    r.state = NUC_LIVE;
    r.b1 = whole ? 1u : (uint32_t)b1;
    r.b2 = whole ? 0u : (uint32_t)(open ? min(b2, max(bz, b1)) : b2);
    r.n1 = start[b1];
    r.r1 = R1;
    r.r2 = R2;
    r.open = open ? 1u : 0u;
    r.q1 = qv[0];
    r.qk = qv[1];
    *out = r;
  }
}

__global__ __launch_bounds__(NR_T) void k_nuc_race(SampleArgs a, NucLayout N) {
  __shared__ __align__(16) uint32_t start[SEL_NB + 4];
  __shared__ uint32_t nc;
  __shared__ float sb[NR_T / WAVE];
  const int row = (int)blockIdx.y, tid = (int)threadIdx.x, lane = lane_id();
  const uint32_t share = blockIdx.x, wid = (uint32_t)__builtin_amdgcn_readfirstlane(tid / WAVE);
  constexpr uint32_t NW = NR_T / WAVE;
  const NucRow *rec = N.row + row;
  const uint4 st = ((const uint4 *)(N.start + (size_t)row * SEL_NB))[tid];
  if (rec->state != NUC_LIVE) return;
  const uint32_t R1 = rec->r1, R2 = rec->r2;
  ((uint4 *)start)[tid] = st;
  if (tid == 0) {
    start[SEL_NB] = (uint32_t)a.vocab;
    nc = 0u;
  }
  __syncthreads();
  /* 64 ranks at a time, with the e of the block's first and last bucket, or of
   * each rank's own where they lie further apart; the blocks to the shares' waves
   * in `unit`s, one round of bucket searches each.  A share's units lie apart: it
   * has surely kept ranks of its own among them, and a best score to measure the
   * ranks near the cut by (a share of the last ranks alone filed too many). */
  const uint32_t nblk = (R2 + WAVE - 1) / WAVE, shares = gridDim.x;
  const uint32_t unit = min(64u, max(1u, (nblk + shares * NW - 1) / (shares * NW)));
  const float *urow = a.u + (size_t)row * a.k;
  /* (the blocks some rank of which can score `reach`; with top_p near 1 or a low
   * T most cannot, whatever their uniforms) */
  auto blocks = [&](float reach, auto &&fn) {
#pragma unroll 1
    for (uint32_t k0 = (wid * shares + share) * unit; k0 < nblk; k0 += NW * shares * unit) {
      const uint32_t rb = min((k0 + (uint32_t)lane) * WAVE, R2 - 1), re = min(rb + WAVE - 1, R2 - 1);
      const int bf = nuc_bucket_of(start, rb), bl = nuc_bucket_of(start, re);
      const float hi = nuc_ehi(bf), lo = nuc_elo(bl);
      const uint32_t kn = min(unit, nblk - k0);
      uint64_t todo = __ballot((uint32_t)lane < kn && hi * ((1.0f + 0x1p-10f) / NU_LEAST) >= reach);
#pragma unroll 1
      while (todo) {
        float u[8];
        int at[8]; /* (uniform) */
#pragma unroll
        for (int j = 0; j < 8; j++) {
          at[j] = todo ? (int)__builtin_ctzll(todo) : -1;
          todo &= todo - 1ull;
          const uint32_t r = (k0 + (uint32_t)at[j]) * WAVE + lane;
          u[j] = at[j] >= 0 && r < R2 ? urow[r] : 2.0f;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
          if (at[j] < 0) break;
          const int l = at[j];
          const uint32_t r = (k0 + (uint32_t)l) * WAVE + lane;
          float h = readlane_f(hi, l), e = readlane_f(lo, l);
          /* (noise is at least u - 2^-24) */
          if (__ballot(u[j] * reach <= h * (1.0f + 0x1p-10f) + reach * 0x1p-23f) == 0ull) continue;
          if (readlane_u((uint32_t)bl, l) - readlane_u((uint32_t)bf, l) > 1u) {
            const int b = nuc_bucket_of(start, min(r, R2 - 1));
            h = nuc_ehi(b);
            e = nuc_elo(b);
          }
          fn(r, u[j], h, e);
        }
      }
    }
  };
  float best = 0.0f;
  auto least = [&](uint32_t r, float u, float, float lo) {
    const float lb = lo * __builtin_amdgcn_rcpf(nuc_noise_hi(u));
    if (r < R1 && nuc_races(u)) best = fmaxf(best, lb);
  };
  auto all_waves = [&]() {
    best = wave_max_f(best);
    if (lane == 0) sb[wid] = best;
    __syncthreads();
#pragma unroll
    for (uint32_t w = 0; w < NW; w++) best = fmaxf(best, sb[w]);
    __syncthreads();
  };
  /* (the first ranks hold much of a peaked row's mass: a share whose own ranks
   * are few or light still has a score to reach) */
  const uint32_t most = min(R1, NU_TOP);
  float ut[NU_TOP / NR_T];
#pragma unroll
  for (uint32_t q = 0; q < NU_TOP / NR_T; q++) ut[q] = tid + q * NR_T < most ? urow[tid + q * NR_T] : 2.0f;
#pragma unroll
  for (uint32_t q = 0; q < NU_TOP / NR_T; q++)
    if (tid + q * NR_T < most) least(tid + q * NR_T, ut[q], 0.0f, nuc_elo(nuc_bucket_of(start, tid + q * NR_T)));
  all_waves();
  blocks(best, least);
  all_waves();
  best *= 1.0f - 0x1p-14f; /* (the reciprocal's error and the scores' own roundings) */
  NucShare *out = N.share + (size_t)row * BK_SMAX + share;
  const bool found = best > 0x1p-100f && best < 0x1p100f;
  if (found) {
    const float inv = __builtin_amdgcn_rcpf(best) * (1.0f + 0x1p-14f);
    blocks(best, [&](uint32_t r, float u, float hi, float) {
      /* u <= -log(1 - u) + 2^-24, so this passes every rank whose score can reach best */
      if (r < R2 && nuc_races(u) && u <= hi * inv * (1.0f + 0x1p-14f) + 0x1p-23f) {
        const int b = nuc_bucket_of(start, r);
        const float nl = nuc_noise_lo(u), eh = nuc_ehi(b);
        if (nl <= eh * inv) {
          const uint32_t s = atomicAdd(&nc, 1u);
          if (s < (uint32_t)NU_C) {
            out->rank[s] = r;
            out->bucket[s] = (uint32_t)b;
            out->start[s] = start[b];
            out->most[s] = nl > 0.0f ? eh * __builtin_amdgcn_rcpf(nl) * (1.0f + 0x1p-14f) : 0x1p120f;
          }
        }
      }
    });
  }
  __syncthreads();
  if (tid == 0) {
    out->best = found ? best : 0.0f;
    out->n = share * unit < nblk && !found ? NU_C + 1u : nc; /* (too many: the row is sorted) */
  }
}

/* the row's candidates: those of its shares' that can reach the row's best.
 * Every wave of the workgroup alike: shares by lane, then fn(share, slot) for
 * each; false when some share had too many. */
template <class Fn>
__device__ __forceinline__ bool nuc_candidates(const NucLayout &N, int row, Fn &&fn) {
  const int lane = lane_id();
  const NucShare *sh = N.share + (size_t)row * BK_SMAX;
  float best = 0.0f;
  uint32_t n = 0u;
  if (lane < N.nseg) {
    best = sh[lane].best;
    n = sh[lane].n;
  }
  best = wave_max_f(best);
  if (__ballot(n > (uint32_t)NU_C)) return false;
  const uint32_t inc = wave_scan_add_u32(n), tot = readlane_u(inc, WAVE - 1);
#pragma unroll 1
  for (uint32_t c0 = 0; c0 < tot; c0 += WAVE) { /* lane l: the shares' candidate c0 + l */
    const uint32_t c = c0 + lane;
    int s = 0;
    for (int q = 0; q < N.nseg; q++) s += readlane_u(inc, q) <= c ? 1 : 0;
    const bool in = c < tot;
    const uint32_t before = (uint32_t)__shfl((int)(inc - n), s); /* (by every lane) */
    const uint32_t slot = in ? c - before : 0u;
    const NucShare *p = sh + (in ? s : 0);
    fn(in && p->most[slot] >= best, p, slot);
  }
  return true;
}

template <bool BF16>
__global__ __launch_bounds__(SEL_T) void k_nuc_gather(SampleArgs a, SelLayout F, NucLayout N) {
  constexpr int EPC = BF16 ? 8 : 4;
  __shared__ uint32_t bits[SEL_NB / 32], na, nb;
  __shared__ uint64_t sum[SEL_NW];
  /* each wave's logits that reach the last bucket wanted, with their positions,
   * taken 64 at a time (most lanes of a chunk hold none) */
  __shared__ uint2 held[SEL_NW][(EPC + 1) * WAVE];
  const int seg = (int)blockIdx.x, row = (int)blockIdx.y, tid = (int)threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = lane_id();
  const SelRun run = sel_run<BF16>(a, F, row, seg, wid);
  uint4 first[SEL_U];
  sel_load(run, run.c0, first);
  const NucRow *rec = N.row + row;
  if (rec->state != NUC_LIVE) return;
  const float M = rec->M, lse = rec->lse;
  const int b1 = (int)rec->b1, b2 = (int)rec->b2;
  const int bsum = b1 <= b2 ? b1 : 0; /* (no cut to find: no sum) */
  if (tid < SEL_NB / 32) bits[tid] = 0u;
  if (tid == 0) na = nb = 0u;
  const RowP rp = row_params(a, row);
  const float T = rp.T, y = 1.0f / T;
  __syncthreads();
  int top = b1 <= b2 ? b2 : 0;
  const bool ok_row = nuc_candidates(N, row, [&](bool in, const NucShare *p, uint32_t slot) {
    const int b = in ? (int)p->bucket[slot] : 0;
    top = max(top, -wave_min_i32(-b));
    if (in && wid == 0) atomicOr(&bits[b >> 5], 1u << (b & 31));
  });
  if (!ok_row) return; /* (the last kernel sorts the row) */
  __syncthreads();
  const float Lc = sel_logit_bound(M, T, top);
  uint64_t *outa = N.keys + (size_t)row * 2 * (size_t)N.vstride + (size_t)seg * N.rstride, *outb = outa + N.vstride;
  uint64_t acc = 0ull;
  uint32_t n = 0u; /* (uniform) logits held */
  auto take = [&](uint32_t from, bool in) {
    const uint2 h = in ? held[wid][from + lane] : make_uint2(0u, 0u);
    const float x = scale_logit(d3s_u2f(h.x), T, y, T < __builtin_inff());
    const int b = sel_bucket(x - M);
    if (in && b < bsum) acc += d3s_fix40_exp(x - lse); /* (x <= m <= lse) */
    const bool ma = in && b >= b1 && b <= b2;
    const bool mb = in && !ma && ((bits[b >> 5] >> (b & 31)) & 1u);
    const uint64_t key = composite_key(x, (int)h.y);
    const int sa = wave_append(ma, (int *)&na);
    if (sa >= 0) outa[sa] = key;
    const int sb = wave_append(mb, (int *)&nb);
    if (sb >= 0) outb[sb] = key;
  };
  sel_chunks<BF16>(run, a.vocab, rp.banned, first, [&](const auto &v, int p0, uint32_t ok) {
    uint32_t m = 0u;
#pragma unroll
    for (int e = 0; e < EPC; e++) m |= (v[e] >= Lc ? 1u : 0u) << e;
    m &= ok;
    if (__ballot(m != 0u) == 0ull) return;
    const uint32_t c = (uint32_t)__popc(m);
    const uint32_t inc = wave_scan_add_u32(c);
    uint32_t s = n + inc - c;
#pragma unroll
    for (int e = 0; e < EPC; e++)
      if ((m >> e) & 1u) held[wid][s++] = make_uint2(d3s_f2u(v[e]), (uint32_t)(p0 + e));
    n += readlane_u(inc, WAVE - 1);
    wave_lds_sync();
#pragma unroll 1
    while (n >= (uint32_t)WAVE) {
      n -= WAVE;
      take(n, true);
    }
    wave_lds_sync();
  });
  if (n > 0u) take(0u, (uint32_t)lane < n);
  acc = wave_sum_mod64(acc);
  if (lane == 0) sum[wid] = acc;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < SEL_NW; w++) acc += sum[w];
    NucSeg &s = N.seg[(size_t)row * BK_SMAX + seg];
    s.na = na;
    s.nb = nb;
    s.psum = acc;
  }
}

/* a gathered set.  Its keys are read 64 consecutive ones of a segment at a time,
 * a wave each, the 64s numbered over the segments: lane s holds how many there
 * are up to segment s, and how many keys s has, so a ballot finds the segment
 * (a search by key in LDS took half of a pass) */
struct NucSet {
  const uint64_t *keys;
  const uint32_t *base; /* LDS: the segments' places, BK_SMAX + 1 */
  int rstride;
  uint32_t n;
  uint32_t upto, count; /* by lane */
  __device__ __forceinline__ uint64_t at(uint32_t i) const {
    int sg = 0;
#pragma unroll
    for (int step = BK_SMAX / 2; step >= 1; step >>= 1) sg += base[sg + step] <= i ? step : 0;
    return keys[(size_t)sg * rstride + (i - base[sg])];
  }
  /* fn(key) for each element, by the whole workgroup */
  template <class Fn>
  __device__ __forceinline__ void each(Fn &&fn) const {
    const int lane = lane_id(), wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
    const uint32_t all = readlane_u(upto, BK_SMAX - 1);
#pragma unroll 1
    for (uint32_t c0 = wid; c0 < all; c0 += 8 * NU_NW) {
      uint64_t kv[8];
      uint32_t in = 0u;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const uint32_t c = c0 + q * NU_NW;
        const int sg = (int)__popcll(__ballot(lane < BK_SMAX && upto <= c)); /* (uniform; BK_SMAX past the last) */
        const uint32_t first = sg ? readlane_u(upto, sg - 1) : 0u;
        const uint32_t i = (c - first) * WAVE + lane;
        const bool ok = c < all && i < readlane_u(count, sg);
        in |= (ok ? 1u : 0u) << q;
        kv[q] = ok ? keys[(size_t)sg * rstride + i] : 0ull;
      }
#pragma unroll
      for (int q = 0; q < 8; q++)
        if ((in >> q) & 1u) fn(kv[q]);
    }
  }
};

struct __align__(16) NucLds {
  uint64_t list[NU_SMALL + 2], ranked[NU_SMALL];
  union {
    struct { /* a large set's counts and sums by 11 bits of what its keys span */
      uint64_t ps[SEL_NB];
      uint32_t hist[SEL_NB];
    };
    struct { /* nuc_sort_row's places by wave and digit */
      uint32_t wcnt[NU_NW][NB], base[NB];
    };
  };
  uint64_t sq[NU_NW], lo, hi, p;
  uint32_t sh[NU_NW], n, above, count;
  int bin;
  uint32_t abase[BK_SMAX + 1], bbase[BK_SMAX + 1];
  uint64_t ckey[WAVE];
  uint32_t crank[WAVE], cbucket[WAVE], cstart[WAVE];
};

/* how far to shift what [0, span] holds for 11 bits of it */
__device__ __forceinline__ int nuc_shift(uint64_t span) {
  return span ? max(0, 64 - (int)__builtin_clzll(span) - 11) : 0;
}

/* the least and greatest val(key) of a set's keys for which in(key); lo > hi:
 * none.  Opens and ends with a barrier. */
template <class In, class Val>
__device__ __forceinline__ void nuc_range(const NucSet &A, NucLds &L, uint64_t &lo, uint64_t &hi, In &&in, Val &&val) {
  __syncthreads();
  if (threadIdx.x == 0) {
    L.lo = ~0ull;
    L.hi = 0ull;
  }
  __syncthreads();
  lo = ~0ull;
  hi = 0ull;
  A.each([&](uint64_t key) {
    if (in(key)) {
      const uint64_t v = val(key);
      lo = v < lo ? v : lo;
      hi = v > hi ? v : hi;
    }
  });
#pragma unroll
  for (int sh = 1; sh < WAVE; sh <<= 1) {
    const uint64_t l2 = (uint64_t)__shfl_xor((unsigned long long)lo, sh), h2 = (uint64_t)__shfl_xor((unsigned long long)hi, sh);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  if (lane_id() == 0 && lo <= hi) { /* (an atomic a wave: 1024 on one word took 9 us) */
    atomicMin((unsigned long long *)&L.lo, (unsigned long long)lo);
    atomicMax((unsigned long long *)&L.hi, (unsigned long long)hi);
  }
  __syncthreads();
  lo = L.lo;
  hi = L.hi;
}

/* the keys of a set for which in(key), at most NU_SMALL of them, ranked;
 * other(key) for the others */
template <class In, class Other>
__device__ __forceinline__ uint32_t nuc_collect(const NucSet &A, NucLds &L, In &&in, Other &&other) {
  __syncthreads();
  if (threadIdx.x == 0) L.n = 0u;
  __syncthreads();
  A.each([&](uint64_t key) {
    if (in(key))
      L.list[atomicAdd(&L.n, 1u)] = key;
    else
      other(key);
  });
  __syncthreads();
  const uint32_t n = L.n;
  rank_by_count<NU_T>(L.list, n, (int)n, L.ranked);
  return n;
}

/* what a search for the cut has behind it: ranks, and their sums of
 * fix40(d3s_expf(x - lse)) (p) and of fix40(d3s_expf(x - m)) (k) */
struct NucSum {
  uint32_t n;
  uint64_t p, k;
};

/* whether a rank r = at.n - 1 that ends with these sums is dropped, or is past k */
__device__ __forceinline__ bool nuc_past(uint32_t n, uint64_t p, uint32_t k, float top_p) {
  return n > k || (n > 1u && d3s_fixsum_to_f32(p) > top_p);
}

/* the cut among the n ranked keys of L.ranked, from `at` on; at: the ranks
 * before the cut and their sums (all of them when it is not there) */
__device__ __forceinline__ bool nuc_cut_small(NucLds &L, uint32_t n, float M, float lse, float top_p, uint32_t k,
                                              NucSum &at) {
  const int tid = (int)threadIdx.x, lane = lane_id(), wid = tid / WAVE;
  const bool in = (uint32_t)tid < n;
  const float x = in ? key_x(L.ranked[tid]) : 0.0f;
  const uint64_t f = in ? d3s_fix40_exp(x - lse) : 0ull;
  uint64_t tot;
  const uint64_t P = at.p + nuc_scan(f, L.sq, tot) + f;
  const uint32_t r = at.n + (uint32_t)tid;
  const int cm = wave_min_i32(in && nuc_past(r + 1u, P, k, top_p) ? (int)r : 0x7fffffff);
  if (lane == 0) L.sh[wid] = (uint32_t)cm;
  __syncthreads();
  uint32_t cut = at.n + n;
#pragma unroll
  for (int w = 0; w < NU_NW; w++) cut = min(cut, L.sh[w]);
  uint64_t ks;
  (void)nuc_scan(in && r < cut ? d3s_fix40_exp(x - M) : 0ull, L.sq, ks);
  const bool hit = cut < at.n + n;
  at.n = cut;
  at.k += ks;
  return hit;
}

/* The same in a large set of the cut's buckets: the range of its order keys;
 * their counts and exact sums by 11 bits of it (the digits of a bucket's few
 * values lie apart, where the key's leading bytes are all the same); the first
 * digit whose last rank is dropped; and so on in that digit until its keys are
 * few (ranked) or equal.  at.k only where the cut is found.  equal: the set's
 * elements all are. */
__device__ __forceinline__ bool nuc_cut_large(const NucSet &A, NucLds &L, float M, float lse, float top_p, uint32_t k,
                                              NucSum &at, bool &equal) {
  const int tid = (int)threadIdx.x, lane = lane_id();
  uint64_t lo, hi;
  nuc_range(A, L, lo, hi, [](uint64_t) { return true; }, [](uint64_t key) { return key >> 32; });
  equal = lo == hi;
  uint32_t count = A.n;
#pragma unroll 1
  while (lo < hi && count > NU_SMALL) {
    const int shift = nuc_shift(hi - lo);
    static_assert(SEL_NB == 2 * NU_T, "a thread two digits");
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; j++) {
      L.hist[tid + j * NU_T] = 0u;
      L.ps[tid + j * NU_T] = 0ull;
    }
    if (tid == 0) L.bin = SEL_NB;
    __syncthreads();
    A.each([&](uint64_t key) {
      const uint32_t o = (uint32_t)(key >> 32);
      if (o >= lo && o <= hi) {
        const int d = (int)((hi - o) >> shift);
        const uint64_t f = d3s_fix40_exp(key_x(key) - lse);
        auto add = [&](uint32_t c) {
          atomicAdd(&L.hist[d], c);
          if (f) atomicAdd((unsigned long long *)&L.ps[d], (unsigned long long)(f * c));
        };
        /* equal elements (rounded logits) by one of their lanes */
        uint64_t left = __ballot(true);
#pragma unroll 1
        for (int t = 0; t < 4 && left; t++) {
          const int l = (int)__builtin_ctzll(left);
          const uint64_t same = __ballot(((left >> lane) & 1ull) && o == readlane_u(o, l));
          if (__popcll(same) < 16) break;
          if (lane == l) add((uint32_t)__popcll(same));
          left &= ~same;
        }
        if ((left >> lane) & 1ull) add(1u);
      }
    });
    __syncthreads();
    const uint2 c = ((const uint2 *)L.hist)[tid];
    const ulonglong2 p = ((const ulonglong2 *)L.ps)[tid];
    uint32_t nb, nt;
    uint64_t pt;
    const uint64_t pb = at.p + nuc_scan2(p.x + p.y, c.x + c.y, L.sq, L.sh, pt, nb, nt);
    nb += at.n;
    const bool past0 = c.x && nuc_past(nb + c.x, pb + p.x, k, top_p);
    const bool past1 = c.y && nuc_past(nb + c.x + c.y, pb + p.x + p.y, k, top_p);
    const int b = wave_min_i32(past0 ? 2 * tid : past1 ? 2 * tid + 1 : SEL_NB);
    if (lane == 0 && b < SEL_NB) atomicMin(&L.bin, b);
    __syncthreads();
    const int bin = L.bin;
    if (bin == SEL_NB) { /* no cut in the set */
      at.n += nt;
      return false;
    }
    if (tid == bin / 2) {
      const bool second = bin & 1;
      L.n = nb + (second ? c.x : 0u);
      L.p = pb + (second ? p.x : 0ull);
      L.count = second ? c.y : c.x;
    }
    __syncthreads();
    at.n = L.n;
    at.p = L.p;
    count = L.count;
    hi -= (uint64_t)bin << shift;
    const uint64_t span = (1ull << shift) - 1ull;
    lo = hi - lo > span ? hi - span : lo;
  }
  /* the kept sum before the keys left, and those ranked, or all of them equal */
  uint64_t above = 0ull, tot;
  auto sum = [&](uint64_t key) { above += (key >> 32) > hi ? d3s_fix40_exp(key_x(key) - M) : 0ull; };
  if (lo < hi) {
    const uint32_t n = nuc_collect(A, L, [&](uint64_t key) { return (key >> 32) >= lo && (key >> 32) <= hi; }, sum);
    (void)nuc_scan(above, L.sq, tot);
    at.k += tot;
    return nuc_cut_small(L, n, M, lse, top_p, k, at);
  }
  if (count < A.n) {
    A.each(sum);
    (void)nuc_scan(above, L.sq, tot);
    at.k += tot;
  }
  /* `count` equal elements: the first rank j of them (not rank 0) past top_p, or rank k */
  const float x = d3s_from_ordkey((uint32_t)hi);
  const uint64_t f = d3s_fix40_exp(x - lse), e = d3s_fix40_exp(x - M), need = d3s_fixsum_gt_threshold(top_p);
  uint64_t j = 0ull;
  if (at.p < need) j = f && need != ~0ull ? (need - at.p + f - 1ull) / f - 1ull : ~0ull;
  if (at.n == 0u && j == 0ull) j = 1ull; /* (rank 0 is kept) */
  if (j > count) j = count;
  if (at.n + (uint32_t)j > k) j = k - at.n;
  at.n += (uint32_t)j;
  at.k += j * e;
  return j < count;
}

/* element j (descending x, then ascending index) of the set's bucket b */
__device__ __forceinline__ uint64_t nuc_select(const NucSet &A, NucLds &L, float M, int b, uint32_t j) {
  const int tid = (int)threadIdx.x;
  auto mine = [&](uint64_t key) { return sel_bucket(key_x(key) - M) == b; };
  uint64_t lo, hi;
  nuc_range(A, L, lo, hi, mine, [](uint64_t key) { return key; });
  uint32_t need = j + 1u;
#pragma unroll 1
  while (lo < hi) { /* (no two keys are equal) */
    const int shift = nuc_shift(hi - lo);
    __syncthreads();
    L.hist[tid] = L.hist[tid + NU_T] = 0u;
    __syncthreads();
    A.each([&](uint64_t key) {
      if (key >= lo && key <= hi && mine(key)) atomicAdd(&L.hist[(hi - key) >> shift], 1u);
    });
    __syncthreads();
    const uint32_t c0 = L.hist[2 * tid], c1 = L.hist[2 * tid + 1];
    uint32_t all;
    const uint32_t before = block_excl_scan_u32<NU_NW>(c0 + c1, L.sh, all);
    if (before < need && before + c0 + c1 >= need) { /* one thread's */
      const bool second = before + c0 < need;
      L.bin = 2 * tid + (second ? 1 : 0);
      L.above = before + (second ? c0 : 0u);
      L.count = second ? c1 : c0;
    }
    __syncthreads();
    const uint64_t top = hi - ((uint64_t)L.bin << shift), span = (1ull << shift) - 1ull;
    const uint32_t count = L.count;
    need -= L.above;
    lo = top - lo > span ? top - span : lo;
    hi = top;
    if (count <= NU_SMALL) {
      (void)nuc_collect(A, L, [&](uint64_t key) { return key >= lo && key <= hi && mine(key); }, [](uint64_t) {});
      return L.ranked[need - 1u];
    }
  }
  return hi;
}

/* whether no rank of the row scores (1 - u, as rounded, is 1, negative or NaN for
 * all: every score counts as -1); by the whole workgroup */
__device__ __forceinline__ bool nuc_none_scores(const SampleArgs &a, int row) {
  const float *u = a.u + (size_t)row * a.k;
  int none = 1;
#pragma unroll 8
  for (int r = (int)threadIdx.x; r < a.k; r += NU_T) {
    const float w = 1.0f - u[r];
    none &= w == 1.0f || !(w >= 0.0f) ? 1 : 0;
  }
  return __syncthreads_and(none) != 0;
}

/* the row's first rank: its greatest composite key */
template <bool BF16>
__device__ __forceinline__ void nuc_first_rank(const SampleArgs &a, int row, NucLds &L, const RowP &rp) {
  const char *rowp = (const char *)a.logits + (size_t)row * (size_t)a.row_stride * (BF16 ? 2 : 4);
  const float y = 1.0f / rp.T;
  uint64_t top = 0ull;
#pragma unroll 8
  for (int i = (int)threadIdx.x; i < a.vocab; i += NU_T) {
    const uint64_t key =
        composite_key(scale_logit(load_logit<BF16>(rowp, i, rp.banned), rp.T, y, rp.T < __builtin_inff()), i);
    top = key > top ? key : top;
  }
#pragma unroll
  for (int sh = 1; sh < WAVE; sh <<= 1) {
    const uint64_t o = (uint64_t)__shfl_xor((unsigned long long)top, sh);
    top = o > top ? o : top;
  }
  if (lane_id() == 0) L.sq[threadIdx.x / WAVE] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
    top = L.sq[0];
    for (int w = 1; w < NU_NW; w++) top = L.sq[w] > top ? L.sq[w] : top;
    a.ids[row] = key_idx(top);
  }
}

/* the row sorted by one workgroup (a stable LSD radix sort by ordkey(x)
 * descending, as k_bk_pass's tiles do it), and the op graph's tail over it: the
 * rare rows nothing else settles */
template <bool BF16>
__device__ __forceinline__ void nuc_sort_row(const SampleArgs &a, int row, const NucLayout &N, NucLds &L, float lse,
                                             const RowP &rp) {
  const int tid = (int)threadIdx.x, lane = lane_id(), wid = tid / WAVE;
  const int V = a.vocab;
  uint64_t *src = N.keys + (size_t)row * 2 * (size_t)N.vstride, *dst = src + N.vstride;
  const char *rowp = (const char *)a.logits + (size_t)row * (size_t)a.row_stride * (BF16 ? 2 : 4);
  const float y = 1.0f / rp.T;
  for (int i = tid; i < V; i += NU_T)
    src[i] = composite_key(scale_logit(load_logit<BF16>(rowp, i, rp.banned), rp.T, y, rp.T < __builtin_inff()), i);
  const uint64_t lt = (1ull << lane) - 1ull;
  uint32_t *base = L.base;
#pragma unroll 1
  for (int pass = 0; pass < 4; pass++) {
    __syncthreads();
    if (tid < NB) base[tid] = 0u;
    for (int i = tid; i < NU_NW * NB; i += NU_T) (&L.wcnt[0][0])[i] = 0u;
    __syncthreads();
    for (int i = tid; i < V; i += NU_T) atomicAdd(&base[bk_digit(src[i], pass)], 1u);
    __syncthreads();
    if (wid == 0) {
      uint32_t h[4], s = 0u;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        h[q] = base[4 * lane + q];
        s += h[q];
      }
      uint32_t at = wave_scan_add_u32(s) - s;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        base[4 * lane + q] = at;
        at += h[q];
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int t0 = 0; t0 < V; t0 += NU_T) {
      const int i = t0 + tid;
      const bool in = i < V;
      const uint64_t key = in ? src[i] : 0ull;
      const uint32_t d = bk_digit(key, pass);
      const uint64_t peers = wave_peers<8>(d, __ballot(in));
      const uint32_t below = (uint32_t)__popcll(peers & lt);
      if (in && below == 0u) L.wcnt[wid][d] = (uint32_t)__popcll(peers);
      __syncthreads();
      if (tid < NB) {
        uint32_t at = base[tid];
        for (int w = 0; w < NU_NW; w++) {
          const uint32_t c = L.wcnt[w][tid];
          L.wcnt[w][tid] = at;
          at += c;
        }
        base[tid] = at;
      }
      __syncthreads();
      if (in) dst[L.wcnt[wid][d] + below] = key;
      __syncthreads();
      for (int j = tid; j < NU_NW * NB; j += NU_T) (&L.wcnt[0][0])[j] = 0u;
      __syncthreads();
    }
    uint64_t *t = src;
    src = dst;
    dst = t;
  }
  __syncthreads();
  generic_tail_opgraph<NU_T>(a, row, lse, rp.top_p, src);
}

/* MINW: waves a SIMD that the registers must allow.  Two workgroups a CU (64
 * registers, the rare paths spilling) when there are more rows than CUs, else
 * one: [2048, 8193] 24.7 us a launch of 1024 rows against 33.4, but [64, 151936]
 * 13.9 against 11.9 us. */
template <bool BF16, int MINW>
__global__ __launch_bounds__(NU_T, MINW) void k_nuc_final(SampleArgs a, NucLayout N) {
  __shared__ __align__(16) NucLds L;
  const int row = (int)blockIdx.x, tid = (int)threadIdx.x, lane = lane_id();
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const NucRow *rec = N.row + row;
  const uint32_t state = rec->state;
  if (state == NUC_REFUSED || state == NUC_MASKED) {
    write_special(a, row, state == NUC_MASKED);
    return;
  }
  const RowP rp = row_params(a, row);
  const float top_p = rp.top_p, M = rec->M, lse = rec->lse;
  const uint32_t k = (uint32_t)a.k;
  {
    const uint32_t b1 = rec->b1, b2 = rec->b2, n1 = rec->n1;
    /* the row's candidates, at most one a lane (every wave files the same) */
    uint32_t ncand = 0u;
    const bool few = nuc_candidates(N, row, [&](bool in, const NucShare *p, uint32_t slot) {
      const uint64_t m = __ballot(in);
      const uint32_t at = ncand + (uint32_t)mbcnt64(m);
      if (in && wid == 0 && at < (uint32_t)WAVE) {
        L.crank[at] = p->rank[slot];
        L.cbucket[at] = p->bucket[slot];
        L.cstart[at] = p->start[slot];
      }
      ncand += (uint32_t)__popcll(m);
    });
    if (!few || ncand > (uint32_t)WAVE) goto sort; /* (uniform) */
    uint32_t cr = 0u, cs = 0u;
    float cu = 0.0f;
    int cb = 0;
    NucSeg sg{};
    if (lane < N.nseg) sg = N.seg[(size_t)row * BK_SMAX + lane];
    const uint32_t ia = wave_scan_add_u32(sg.na), ib = wave_scan_add_u32(sg.nb);
    if (wid == 0) {
      if (lane < BK_SMAX) {
        L.abase[lane + 1] = ia;
        L.bbase[lane + 1] = ib;
      }
      if (lane == 0) L.abase[0] = L.bbase[0] = 0u;
    }
    const uint64_t P1 = wave_sum_mod64(sg.psum);
    __syncthreads();
    if ((uint32_t)lane < ncand) { /* lane c's candidate: rank, uniform, bucket and its first rank */
      cr = L.crank[lane];
      cb = (int)L.cbucket[lane];
      cs = L.cstart[lane];
      cu = a.u[(size_t)row * a.k + cr];
    }
    const uint64_t *keys = N.keys + (size_t)row * 2 * (size_t)N.vstride;
    const NucSet A{keys, L.abase, N.rstride, L.abase[BK_SMAX], wave_scan_add_u32((sg.na + WAVE - 1) / WAVE), sg.na};
    const NucSet B{keys + N.vstride, L.bbase, N.rstride, L.bbase[BK_SMAX], wave_scan_add_u32((sg.nb + WAVE - 1) / WAVE),
                   sg.nb};

    /* ---- the cut and the kept sum */
    uint32_t cut = k;
    uint64_t kept = rec->qk;
    const bool small_a = A.n <= NU_SMALL;
    bool whole_row = false; /* the row's elements are all equal: rank r is element r */
    if (b1 <= b2) {
      NucSum at{n1, P1, rec->q1};
      bool hit, equal = false;
      if (small_a) {
        if ((uint32_t)tid < A.n) L.list[tid] = A.at((uint32_t)tid);
        __syncthreads();
        rank_by_count<NU_T>(L.list, A.n, (int)A.n, L.ranked);
        hit = nuc_cut_small(L, A.n, M, lse, top_p, k, at);
      } else {
        hit = nuc_cut_large(A, L, M, lse, top_p, k, at, equal);
        whole_row = equal && A.n == (uint32_t)a.vocab;
      }
      if (hit || !rec->open) {
        cut = min(k, at.n);
        kept = at.k;
      }
    }

    /* ---- the candidates' elements */
    if (small_a && wid == 0 && (uint32_t)lane < ncand && cr >= n1 && cr - n1 < A.n) L.ckey[lane] = L.ranked[cr - n1];
    __syncthreads();
    const bool small_b = B.n <= NU_SMALL;
    if (small_b && B.n > 0u) {
      if ((uint32_t)tid < B.n) L.list[tid] = B.at((uint32_t)tid);
      __syncthreads();
      rank_by_count<NU_T>(L.list, B.n, (int)B.n, L.ranked);
    }
    /* (A: the ranks from n1 on, b1 <= b2) */
    if (small_b)
      for (uint32_t c = wid; c < ncand; c += NU_NW) {
        const uint32_t r = readlane_u(cr, (int)c), s = readlane_u(cs, (int)c);
        const int b = (int)readlane_u((uint32_t)cb, (int)c);
        if (r >= n1 && r - n1 < A.n) continue;
        /* its bucket's elements are consecutive in the sorted set */
        uint32_t before = 0u;
        for (uint32_t i = lane; i - lane < B.n; i += WAVE)
          before += (uint32_t)__popcll(__ballot(i < B.n && sel_bucket(key_x(L.ranked[min(i, B.n - 1u)]) - M) < b));
        if (lane == 0) L.ckey[c] = L.ranked[min(before + (r - s), NU_SMALL - 1u)];
      }
    for (uint32_t c = 0; c < ncand; c++) { /* (uniform; nuc_select takes L.ranked over) */
      const uint32_t r = readlane_u(cr, (int)c), s = readlane_u(cs, (int)c);
      const bool in_a = r >= n1 && r - n1 < A.n;
      if (in_a ? small_a : small_b) continue;
      NucSet S = A;
      if (!in_a) S = B;
      const uint64_t key = whole_row ? composite_key(M, (int)r)
                                     : nuc_select(S, L, M, (int)readlane_u((uint32_t)cb, (int)c), r - s);
      if (tid == 0) L.ckey[c] = key;
    }
    __syncthreads();

    /* ---- their scores; the first maximum */
    float sc = -2.0f;
    int rk = 0x7fffffff;
    uint64_t key = 0ull;
    if ((uint32_t)lane < ncand && cr < cut) {
      key = L.ckey[lane];
      const float inv = 1.0f / d3s_fixsum_to_f32(kept);
      const float p = d3s_expf_nonpos(key_x(key) - M) * inv;
      const float score = p / -d3s_logf(1.0f - cu);
      sc = score > -1.0f ? score : -1.0f;
      rk = (int)cr;
    }
    float bs = sc;
    int br = rk;
    wave_argmax(bs, br);
    if (bs > 0.0f) {
      if (wid == 0 && rk == br) a.ids[row] = key_idx(key);
      return;
    }
  }
sort:
  __syncthreads();
  if (nuc_none_scores(a, row)) {
    nuc_first_rank<BF16>(a, row, L, rp);
    return;
  }
  nuc_sort_row<BF16>(a, row, N, L, lse, rp);
}

size_t nuc_row_bytes(const SelLayout &F) {
  return 2 * (size_t)F.vstride * 8u + sizeof(NucRow) + BK_SMAX * (sizeof(NucSeg) + sizeof(NucShare)) + SEL_NB * 4u +
         sel_front_bytes(F, true);
}

}  // namespace

bool nucleus_takes(const SampleArgs &a) {
  return a.opgraph && !a.probs && !a.cand && a.k > SEL_MAX_K && a.vocab > topp_max_vocab();
}

size_t nucleus_workspace_bytes(const SampleArgs &a, Dtype dt, bool one_row) {
  SelLayout F{};
  sel_front_shape(F, a, dt, one_row ? 1 : a.n_rows);
  const size_t row = nuc_row_bytes(F);
  if (one_row) return row;
  const size_t all = row * (size_t)a.n_rows;
  return all <= SEL_WS_CAP ? all : (SEL_WS_CAP > row ? SEL_WS_CAP : row);
}

bool launch_nucleus(const SampleArgs &a, Dtype dt, void *ws, size_t ws_bytes, hipStream_t s) {
  if (!ws || !nucleus_takes(a)) return false;
  int64_t chunk = a.n_rows < 32768 ? a.n_rows : 32768; /* (a grid's second dimension) */
  SelLayout F{};
  for (;; chunk = (chunk + 1) / 2) {
    sel_front_shape(F, a, dt, chunk);
    if (nuc_row_bytes(F) * (size_t)chunk <= ws_bytes) break;
    if (chunk == 1) return false;
  }
  /* against the streaming kernel, or beyond its k the sorting kernels in the same
   * memory (a round of one row: 39 us at V = 20 000, 98 us at 151 936; 64 rows
   * there 167 us).  Here a round of one row takes 34 and 42 us, 64 rows 60 us. */
  const int64_t groups = (a.n_rows + chunk - 1) / chunk;
  if (a.k <= generic_max_k()) {
    if (!rounds_pay(a, groups, 45.0, 6e-6, generic_us(a, dt))) return false;
  } else {
    /* a few short bf16 rows, none of whose ranks top_p drops, at T = 1: two passes
     * sort them, and the search near a prefix of 1 costs more ([1, 17000] 40 us
     * against 44 us, [16, 20000] 47 against 52, [4, 32768] 50 against 53; at 50 000
     * 51 us either way; fp32, four passes, [1, 20000] 58 against 49) */
    if (dt == DT_BF16 && !a.temperature && a.temperature_scalar == 1.0f && !a.top_p && a.top_p_scalar >= 1.0f &&
        a.vocab <= 40000 && a.n_rows <= 32)
      return false;
    const int64_t sorted = std::max<int64_t>(1, (int64_t)(ws_bytes / bigk_row_bytes(a)));
    const double sort_us = (double)((a.n_rows + sorted - 1) / sorted) * (30.0 + 4.5e-4 * a.vocab);
    if (!rounds_pay(a, groups, 45.0, -3e-6, sort_us)) return false; /* (4 against 7 ps an element) */
  }
  for (int64_t r0 = 0; r0 < a.n_rows; r0 += chunk) {
    const int64_t n = a.n_rows - r0 < chunk ? a.n_rows - r0 : chunk;
    const SampleArgs c = rows_from(a, dt, r0, n);
    NucLayout N{};
    N.vstride = F.vstride;
    N.nseg = F.nseg;
    N.rstride = F.segc * (dt == DT_F32 ? 4 : 8);
    N.keys = (uint64_t *)ws;
    F.csum = N.keys + (size_t)n * 2 * (size_t)N.vstride;
    F.cnt = (uint32_t *)(F.csum + (size_t)n * F.nseg * SEL_NB);
    N.start = F.cnt + (size_t)n * F.nseg * SEL_NB; /* (16-byte loads) */
    F.seg = (SelSeg *)(N.start + (size_t)n * SEL_NB);
    N.seg = (NucSeg *)(F.seg + (size_t)n * SEL_SMAX);
    N.row = (NucRow *)(N.seg + (size_t)n * BK_SMAX);
    N.share = (NucShare *)(N.row + n);
    launch_select_front(c, dt, nullptr, F, s);
    const dim3 grid((unsigned)F.nseg, (unsigned)n);
    hipLaunchKernelGGL(k_nuc_bound, dim3((unsigned)n), dim3(NU_T), 0, s, c, F, N);
    hipLaunchKernelGGL(k_nuc_race, grid, dim3(NR_T), 0, s, c, N);
    const bool f32 = dt == DT_F32, two = n > 256;
    if (f32)
      hipLaunchKernelGGL(k_nuc_gather<false>, grid, dim3(SEL_T), 0, s, c, F, N);
    else
      hipLaunchKernelGGL(k_nuc_gather<true>, grid, dim3(SEL_T), 0, s, c, F, N);
    const auto last = f32 ? (two ? k_nuc_final<false, 8> : k_nuc_final<false, 4>)
                          : (two ? k_nuc_final<true, 8> : k_nuc_final<true, 4>);
    hipLaunchKernelGGL(last, dim3((unsigned)n), dim3(NU_T), 0, s, c, N);
  }
  return true;
}

}  // namespace d3s
