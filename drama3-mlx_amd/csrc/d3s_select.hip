/* The selecting path: k beyond one wave (65 .. SEL_MAX_K) on rows longer than
 * the nucleus kernel takes, and smaller k on rows wider than the segmented
 * kernel's (gfx950, wave64).  The op graph's order (src/sampling.c:22-49).
 *
 * A row is cut into segments, a workgroup each, so that a few rows fill the
 * chip, and read three times (once from HBM, then from the caches):
 *  k_sel_max: each segment's largest logit (so m = max x, division being
 *     monotone);
 *  k_sel_hist: every x = L / T exactly and its bucket below the max
 *     (sel_rank_bucket: of a logit's distance, or its relative width; for the
 *     wide nucleus path 1/64 of x, the last one open), counted in LDS and stored
 *     per segment
 *     (adding the segments' counts to one table by global atomics took 6.6 us
 *     more, at [32, 151936]); the segment's exact sum of fix40(d3s_expf(x - m));
 *  k_sel_gather: the first bucket at which the row's count reaches k, by groups
 *     of buckets and then within one; the logits that can lie in it or above
 *     (few more than k), each segment's in a region of its own;
 *  k_sel_sort (a workgroup per row): those logits as composite keys, into LDS
 *     by bucket, each key's rank from the larger keys of its own bucket (or, with
 *     many in one, a radix sort), then the op graph's tail with lse from the
 *     segments' sums.
 * Where the k-th element's bucket holds more than LDS does (masked logits, equal
 * rows: ties by the thousand), it is left out of the gathered keys and
 * k_sel_sort's workgroup finds its first elements in the row (sel_crowd).
 * The sorting path (d3s_bigk.hip) takes the first three as its front.  Every
 * result is the oracle's bits.
 *
 * Bound: latency (four launches; k_sel_sort is one workgroup's chain).
 * [32, 151936] bf16, k = 1000: 3.9 + 8.2 + 8.4 + 13.6 us against 436 us for
 * k_generic, one workgroup a row (T = 1e-5: 33 us a call against 418); [1, 8193], k
 * = 65: 19.6 us against 35.5 us; [2048, 32768], k = 4096: 384 us against 781 us. */
#include <atomic>

#include "d3s_rowcore.h"
#include "d3s_select.h"

#pragma clang fp contract(off)

namespace d3s {
namespace {

constexpr int SEL_CAP = 8192; /* keys k_sel_sort ranks */
/* comparisons a thread makes where keys are ranked by all pairs of a bucket (the
 * most crowded one's keys, for each of its own); past that all go through
 * sel_radix (rounded and quantised logits).  us a call, bf16: [512, 20000], k =
 * 4096, whole numbers: 1043 by pairs, 100 by the radix sort; [32, 151936], k =
 * 4096, eighths: 98 and 48.5; k = 1000, eighths, below the line: 38.5 and 41.6;
 * [1024, 20000], k = 4096, text, below it: 139 and 157. */
constexpr uint32_t SEL_PAIRS = 384;

template <bool BF16>
__global__ __launch_bounds__(SEL_T) void k_sel_max(SampleArgs a, SelLayout L) {
  __shared__ float sh[SEL_NW];
  __shared__ uint32_t shn[SEL_NW];
  const int seg = (int)blockIdx.x, row = (int)blockIdx.y;
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  const SelRun run = sel_run<BF16>(a, L, row, seg, wid);
  uint4 first[SEL_U];
  sel_load(run, run.c0, first);
  const int banned = a.banned ? a.banned[row] : -1;
  const float ninf = -__builtin_inff();
  const float T = a.temperature ? a.temperature[row] : a.temperature_scalar;
  const bool flat = !(T < __builtin_inff()); /* (only T = +inf asks whether some logit is -inf) */
  float m = ninf;
  uint32_t masked = 0u;
  sel_chunks<BF16>(run, a.vocab, banned, first, [&](const auto &v, int, uint32_t ok) {
    constexpr int EPC = BF16 ? 8 : 4;
#pragma unroll
    for (int e = 0; e < EPC; e++) m = fmaximum(m, v[e]);
    if (flat) {
#pragma unroll
      for (int e = 0; e < EPC; e++) masked |= v[e] == ninf ? (ok >> e) & 1u : 0u;
    }
  });
  m = wave_maximum_f(m);
  masked = __ballot(masked != 0u) ? 1u : 0u;
  if (lane_id() == 0) {
    sh[wid] = m;
    shn[wid] = masked;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < SEL_NW; w++) {
      m = fmaximum(m, sh[w]);
      masked |= shn[w];
    }
    SelSeg &sg = L.seg[(size_t)row * SEL_SMAX + seg];
    sg.lmax = m;
    sg.masked = masked;
  }
}

/* SUMS: each bucket's exact sum as well (for the wide nucleus path) */
template <bool BF16, bool SUMS>
__global__ __launch_bounds__(SEL_T) void k_sel_hist(SampleArgs a, SelLayout L) {
  __shared__ __align__(16) uint32_t cnt[SEL_NB];
  __shared__ __align__(16) uint64_t bsum[SUMS ? SEL_NB : 2];
  __shared__ uint64_t sum[SEL_NW];
  constexpr int PER = SEL_NB / SEL_T;
  static_assert(PER == 4 && SEL_G % PER == 0, "a thread's buckets are 16 bytes of one group");
  const int seg = (int)blockIdx.x, row = (int)blockIdx.y, tid = (int)threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const SelRun run = sel_run<BF16>(a, L, row, seg, wid);
  uint4 first[SEL_U];
  sel_load(run, run.c0, first);
  const RowP rp = row_params(a, row);
  const float T = rp.T, y = 1.0f / T;
  ((uint4 *)cnt)[tid] = make_uint4(0u, 0u, 0u, 0u);
  if (SUMS) {
    ((uint4 *)bsum)[2 * tid] = make_uint4(0u, 0u, 0u, 0u);
    ((uint4 *)bsum)[2 * tid + 1] = make_uint4(0u, 0u, 0u, 0u);
  }
  float M;
  if (sel_row_max(L, row, T, M) != SEL_LIVE) return;
  __syncthreads();
  const bool te = sel_t_easy(T);
  const float s = sel_rank_scale(T);
  uint64_t acc = 0ull;
  sel_chunks<BF16>(run, a.vocab, rp.banned, first, [&](const auto &v, int, uint32_t ok) {
    constexpr int EPC = BF16 ? 8 : 4;
    float x[EPC];
    sel_scale(v, T, y, te, x);
    if (SUMS) { /* nearly equal rows: the lanes' equal elements added by one of them */
      const float v0 = readlane_f(v[0], 0);
      if (__popcll(__ballot(v[0] == v0)) > WAVE / 2) {
        const float z0 = readlane_f(x[0], 0) - M;
        const int b0 = sel_bucket(z0);
        uint32_t same = 0u;
#pragma unroll
        for (int e = 0; e < EPC; e++) {
          const bool eq = ((ok >> e) & 1u) && d3s_f2u(x[e]) == d3s_f2u(readlane_f(x[0], 0));
          same += (uint32_t)__popcll(__ballot(eq));
          ok &= ~((eq ? 1u : 0u) << e);
        }
        if (lane_id() == 0 && same && b0 < SEL_NB - 1) {
          atomicAdd(&cnt[b0], same);
          atomicAdd((unsigned long long *)&bsum[b0], (unsigned long long)(d3s_fix40_exp(z0) * same));
        }
      }
    }
#pragma unroll
    for (int e = 0; e < EPC; e++) {
      const float z = x[e] - M;
      const int b = SUMS ? sel_bucket(z) : sel_rank_bucket(z, s);
      /* (the last bucket, where a row's masked or far elements all lie, and those
       * outside the row, has no terms, and its count, kept as 0, is what the others
       * leave of the row: no atomics on one word) */
      if (SUMS) {
        if (((ok >> e) & 1u) && b < SEL_NB - 1) {
          atomicAdd(&cnt[b], 1u);
          atomicAdd((unsigned long long *)&bsum[b], (unsigned long long)d3s_fix40_exp(z));
        }
      } else {
        if (b < SEL_NB - 1) atomicAdd(&cnt[b], 1u);
        acc += d3s_fix40_exp(z);
      }
    }
  });
  const size_t at = (size_t)row * L.nseg + seg;
  if (SUMS) {
    __syncthreads();
    const ulonglong2 p = ((const ulonglong2 *)bsum)[2 * tid], q = ((const ulonglong2 *)bsum)[2 * tid + 1];
    ulonglong2 *out = (ulonglong2 *)(L.csum + at * SEL_NB);
    out[2 * tid] = p;
    out[2 * tid + 1] = q;
    acc = p.x + p.y + q.x + q.y;
  }
  acc = wave_sum_mod64(acc);
  if (lane_id() == 0) sum[wid] = acc;
  __syncthreads();
  const uint4 c = ((const uint4 *)cnt)[tid];
  ((uint4 *)(L.cnt + at * SEL_NB))[tid] = c;
  uint32_t g = c.x + c.y + c.z + c.w; /* (the group's count; the wide nucleus path takes none) */
  g += dpp_u<0xb1, 0xf>(0u, g);   /* quad_perm [1,0,3,2] */
  g += dpp_u<0x4e, 0xf>(0u, g);   /* quad_perm [2,3,0,1] */
  g += dpp_u<0x141, 0xf>(0u, g);  /* row_half_mirror: the other four of the eight */
  if (!SUMS && tid % (SEL_G / PER) == 0) L.group[at * SEL_NG + tid / (SEL_G / PER)] = g;
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < SEL_NW; w++) acc += sum[w];
    L.seg[(size_t)row * SEL_SMAX + seg].sum = acc;
  }
}

/* SORT: the sorting path's front (B): composite keys with their digits' counts */
template <bool BF16, bool SORT>
__global__ __launch_bounds__(SEL_T) void k_sel_gather(SampleArgs a, SelLayout L, BkLayout B) {
  __shared__ uint32_t part[SEL_NW][SEL_NG], fine[SEL_G], wn[SEL_NW];
  __shared__ uint32_t dig[SORT ? 2 : 1][NB], wor[SEL_NW], wand[SEL_NW], wlow[SEL_NW];
  static_assert(SEL_NG == WAVE && SEL_SMAX % SEL_NW == 0, "a lane a group");
  constexpr int EPC = BF16 ? 8 : 4, SM = SORT ? BK_SMAX : SEL_SMAX;
  constexpr int GL = SM / SEL_NW, FL = (SM * SEL_G + SEL_T - 1) / SEL_T;
  const int seg = (int)blockIdx.x, row = (int)blockIdx.y, tid = (int)threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = lane_id();
  const SelRun run = sel_run<BF16>(a, L, row, seg, wid);
  uint4 first[SEL_U];
  sel_load(run, run.c0, first);
  /* the groups' counts: wave w the segments w, w + 8, ... */
  const size_t at0 = (size_t)row * L.nseg;
  uint32_t g[GL];
#pragma unroll
  for (int q = 0; q < GL; q++) {
    const int s = wid + q * SEL_NW;
    g[q] = s < L.nseg ? L.group[(at0 + s) * SEL_NG + lane] : 0u;
  }
  const RowP rp = row_params(a, row);
  const float T = rp.T, y = 1.0f / T;
  float M;
  const SelRow what = sel_row_max(L, row, T, M);
  uint32_t *hx = nullptr, *gh = nullptr;
  if (SORT) { /* the passes' counts: this segment's of digits 0 and 2 below; the later ones are added to */
    gh = B.hist + (size_t)row * 4 * BK_SMAX * NB;
    hx = B.hidx + (size_t)row * 2 * BK_SMAX * NB;
    if (tid < NB) {
      dig[0][tid] = 0u;
      dig[SORT ? 1 : 0][tid] = 0u;
#pragma unroll
      for (int p = 1; p < 4; p++) gh[(p * BK_SMAX + seg) * NB + tid] = 0u;
    }
    if (what != SEL_LIVE && tid == 0) {
      BkMeta m{};
      m.max = what == SEL_MASKED ? -__builtin_inff() : 0.0f;
      m.flags = what == SEL_REFUSED ? 1u : 0u;
      B.meta[(size_t)row * BK_SMAX + seg] = m;
    }
  }
  if (what != SEL_LIVE) return;
  const uint32_t k = (uint32_t)a.k;
#pragma unroll
  for (int q = 1; q < GL; q++) g[0] += g[q];
  part[wid][lane] = g[0];
  if (tid < SEL_G) fine[tid] = 0u;
  __syncthreads();
  uint32_t gt = 0u;
#pragma unroll
  for (int w = 0; w < SEL_NW; w++) gt += part[w][lane];
  const uint32_t gin = wave_scan_add_u32(gt);
  const int tg = (int)__builtin_ctzll(__ballot(gin >= k) | (1ull << (WAVE - 1))); /* the k-th element's group */
  const uint32_t before = readlane_u(gin - gt, tg);
  /* that group's buckets, over the segments */
  uint32_t f = 0u;
#pragma unroll
  for (int q = 0; q < FL; q++) {
    const int s = tid / SEL_G + q * (SEL_T / SEL_G);
    const size_t at = (at0 + s) * SEL_NB + tg * SEL_G + tid % SEL_G;
    f += s < L.nseg ? L.cnt[at] : 0u;
  }
  if (f) atomicAdd(&fine[tid % SEL_G], f);
  __syncthreads();
  const uint32_t fin = before + wave_scan_add_u32(lane < SEL_G ? fine[lane] : 0u);
  const int tb = tg * SEL_G + (int)__builtin_ctzll(__ballot(fin >= k) | (1ull << (SEL_G - 1)));
  /* (a few elements below bucket tb may reach Lc as well, none below Lc's own
   * bucket: the set holds every element above any of its own, which is all that
   * the ranking asks.  Where it may be more than k_sel_sort ranks, the buckets up
   * to tb exactly; where bucket tb alone makes it so, without that one) */
  const float s = sel_rank_scale(T);
  float Lc = sel_rank_bound(M, T, y, tb);
  bool crowd = false;
  if (!SORT) {
    const int at_b = tb - tg * SEL_G;
    const uint32_t next =
        at_b + 1 < SEL_G ? readlane_u(fin, min(at_b + 1, SEL_G - 1)) : readlane_u(gin, min(tg + 1, WAVE - 1));
    const float xc = Lc * y; /* (a little below Lc / T) */
    const int reach = sel_rank_bucket(fminf(xc - fabsf(xc) * 0x1p-20f - M, 0.0f), s);
    /* (the last bucket's elements are not in the counts; a scalar branch lets the
     * rare path lie out of line) */
    const int rare = next > (uint32_t)SEL_CAP || reach > tb + 1 || tb + 2 >= SEL_NB ? 1 : 0;
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(rare) != 0, 0)) {
      crowd = tb == SEL_NB - 1 || readlane_u(fin, at_b) > (uint32_t)SEL_CAP;
      Lc = sel_rank_least(M, T, y, s, crowd ? tb - 1 : tb);
    }
  }
  auto pick = [&](const auto &v, uint32_t ok) -> uint32_t {
    uint32_t m = 0u;
#pragma unroll
    for (int e = 0; e < EPC; e++) m |= (v[e] >= Lc ? 1u : 0u) << e;
    return m & ok;
  };
  uint32_t n = 0u;
  sel_chunks<BF16>(run, a.vocab, rp.banned, first,
                   [&](const auto &v, int, uint32_t ok) { n += (uint32_t)__popc(pick(v, ok)); });
  n = wave_sum_u32(n);
  if (lane == 0) wn[wid] = n;
  __syncthreads();
  uint32_t at = 0u, tot = 0u;
#pragma unroll
  for (int w = 0; w < SEL_NW; w++) {
    at += w < wid ? wn[w] : 0u;
    tot += wn[w];
  }
  if (!SORT) {
    if (tid == 0) {
      SelSeg &sg = L.seg[(size_t)row * SEL_SMAX + seg];
      sg.count = tot;
      sg.crowd = crowd ? (uint32_t)tb + 1u : 0u;
      sg.least = Lc;
    }
    if (n == 0u) return;
  }
  uint64_t *out = SORT ? B.keys + (size_t)row * 2 * (size_t)B.vstride + (size_t)seg * B.rstride
                       : L.keys + (size_t)row * (size_t)L.vstride + (size_t)seg * L.segc * EPC;
  const bool te = sel_t_easy(T);
  uint32_t wo = 0u, wa = ~0u, wl = 0u;
  sel_chunks<BF16>(run, a.vocab, rp.banned, first, [&](const auto &v, int p0, uint32_t ok) {
    const uint32_t m = pick(v, ok);
    if (__ballot(m != 0u) == 0ull) return;
    const uint32_t c = (uint32_t)__popc(m);
    const uint32_t inc = wave_scan_add_u32(c);
    uint32_t slot = at + inc - c;
    if (SORT) {
      float x[EPC];
      sel_scale(v, T, y, te, x);
#pragma unroll
      for (int e = 0; e < EPC; e++)
        if ((m >> e) & 1u) {
          const uint64_t key = composite_key(x[e], p0 + e);
          out[slot++] = key;
          /* (with pass 0 not launched its counts are not read; its digit is
           * then one of two values by the sign: 1024 atomics on two words) */
          if (B.pass0 == 0) atomicAdd(&dig[0][bk_digit(key, 0)], 1u);
          atomicAdd(&dig[SORT ? 1 : 0][bk_digit(key, 2)], 1u);
          const uint32_t dw = (uint32_t)((~key) >> 32); /* the digit word */
          wo |= dw;
          wa &= dw;
          wl |= d3s_f2u(x[e]) & 0xffffu;
        }
    } else {
#pragma unroll
      for (int e = 0; e < EPC; e++)
        if ((m >> e) & 1u) out[slot++] = ((uint64_t)d3s_f2u(v[e]) << 32) | (uint32_t)(p0 + e);
    }
    at += readlane_u(inc, 63);
  });
  if (!SORT) return;
#pragma unroll
  for (int sh = 1; sh < WAVE; sh <<= 1) {
    wo |= (uint32_t)__shfl_xor((int)wo, sh);
    wa &= (uint32_t)__shfl_xor((int)wa, sh);
    wl |= (uint32_t)__shfl_xor((int)wl, sh);
  }
  if (lane == 0) {
    wor[wid] = wo;
    wand[wid] = wa;
    wlow[wid] = wl;
  }
  __syncthreads();
  if (tid < NB) {
    hx[seg * NB + tid] = dig[0][tid];
    hx[(BK_SMAX + seg) * NB + tid] = dig[SORT ? 1 : 0][tid];
  }
  if (tid == 0) {
    BkMeta m{};
    m.max = M;
    m.sum = L.seg[(size_t)row * SEL_SMAX + seg].sum;
    m.kand = ~0u;
#pragma unroll
    for (int w = 0; w < SEL_NW; w++) {
      m.kor |= wor[w];
      m.kand &= wand[w];
      m.klow |= wlow[w];
    }
    m.count = tot;
    B.meta[(size_t)row * BK_SMAX + seg] = m;
  }
}

/* the op graph's tail (generic_tail_opgraph's definition) over k <= NQ GBLOCK
 * ranked keys, thread t holding ranks t NQ .. t NQ + NQ - 1 and their uniforms
 * u */
template <int NQ>
__device__ __forceinline__ void sel_tail(const SampleArgs &a, int row, float lse, float top_p, const uint64_t *ranked,
                                         const float (&u)[NQ]) {
  __shared__ uint32_t sh_u32[GNW], sh_lo[GNW], sh_hi[GNW];
  __shared__ float sh_best[GNW];
  __shared__ int sh_bestr[GNW];
  const int tid = (int)threadIdx.x, lane = lane_id(), wid = tid / WAVE;
  const int k = a.k, r0 = tid * NQ;
  const float v0 = key_x(ranked[0]);
  uint64_t key[NQ], f[NQ], P = 0ull;
  float ex[NQ], noise[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const bool in = r0 + q < k;
    key[q] = in ? ranked[r0 + q] : 0ull;
    f[q] = in ? d3s_fix40_exp(key_x(key[q]) - lse) : 0ull; /* (x <= m <= lse) */
    ex[q] = in ? d3s_expf_nonpos(key_x(key[q]) - v0) : 0.0f;
    noise[q] = -d3s_logf(1.0f - u[q]);
    P += f[q];
  }
  P = block_excl_scan_u64<GNW>(P, sh_lo, sh_hi);
  int cut = k;
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    P += f[q];
    if (r0 + q < k && r0 + q > 0 && cut == k && d3s_fixsum_to_f32(P) > top_p) cut = r0 + q;
  }
  cut = wave_min_i32(cut);
  if (lane == 0) sh_u32[wid] = (uint32_t)cut;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < GNW; w++) cut = min(cut, (int)sh_u32[w]);
  uint64_t ks = 0ull;
#pragma unroll
  for (int q = 0; q < NQ; q++) ks += r0 + q < cut ? d3s_fix40_unit(ex[q]) : 0ull; /* (cut <= k) */
  ks = wave_sum_u64(ks);
  if (lane == 0) {
    sh_lo[wid] = (uint32_t)ks;
    sh_hi[wid] = (uint32_t)(ks >> 32);
  }
  __syncthreads();
  uint64_t KS = 0ull;
#pragma unroll
  for (int w = 0; w < GNW; w++) KS += ((uint64_t)sh_hi[w] << 32) | sh_lo[w];
  const float inv = 1.0f / d3s_fixsum_to_f32(KS);
  float bs = -1.0f;
  int br = 0x7fffffff;
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int r = r0 + q;
    if (r < k) {
      const float p = r < cut ? ex[q] * inv : 0.0f;
      const float score = p / noise[q];
      const float sc = score > -1.0f ? score : -1.0f;
      if (sc > bs || br == 0x7fffffff) { /* first maximum within the thread's ranks */
        bs = sc;
        br = r;
      }
      if (a.probs) a.probs[(size_t)row * k + r] = p;
      if (a.cand) a.cand[(size_t)row * k + r] = key_idx(key[q]);
    }
  }
  wave_argmax(bs, br);
  if (lane == 0) {
    sh_best[wid] = bs;
    sh_bestr[wid] = br;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < GNW; w++)
      if (sh_best[w] > bs || (sh_best[w] == bs && sh_bestr[w] < br)) {
        bs = sh_best[w];
        br = sh_bestr[w];
      }
    a.ids[row] = key_idx(ranked[br]);
  }
}

struct CrowdLds {
  uint32_t lo, hi, n, bin, above, count;
};

/* ranked[n .. k): the rest of the first k, from bucket tb, whose elements are
 * not gathered: the row read again by the whole workgroup, in whole chunks, for
 * the range of the bucket's order keys, for their counts by 11 bits of it until
 * the last rank's is met (one range where all are equal, as masked logits are),
 * and for those above; the equal ones in index order.  Bound: one CU's reads of
 * the row (a 16-byte load a lane) and its scaling: [32, 151936] bf16, k = 1000,
 * all but 60 logits masked: 82 us a call, 138 us for fp32 masked by finite values
 * (773 and 763 us when such a row began again with the generic procedure, 695 and
 * 700 us by the streaming kernel).  list: LDS for the keys, hist: SEL_NB counts, sh: GNW words. */
template <bool BF16>
__device__ __forceinline__ void sel_crowd(const SampleArgs &a, int row, const RowP &rp, float M, int tb, uint32_t n,
                                          uint64_t *ranked, uint64_t *list, uint32_t *hist, uint32_t *sh) {
  constexpr int ES = BF16 ? 2 : 4, EPC = 16 / ES, TIE = 8; /* elements a thread looks at for equal ones */
  __shared__ CrowdLds S;
  const int tid = (int)threadIdx.x, wid = __builtin_amdgcn_readfirstlane(tid / WAVE), V = a.vocab;
  const float T = rp.T, y = 1.0f / T, s = sel_rank_scale(T);
  const bool te = sel_t_easy(T);
  const char *rowp = (const char *)a.logits + (size_t)row * (size_t)a.row_stride * ES;
  SelRun r;
  r.off = (int)(((uintptr_t)rowp & 15u) / ES);
  r.src = (const uint4 *)(rowp - r.off * ES);
  const int nchunks = (r.off + V + EPC - 1) / EPC, wch = (nchunks + GNW - 1) / GNW;
  r.c0 = min(nchunks, wid * wch);
  r.c1 = min(nchunks, r.c0 + wch);
  auto each = [&](auto &&fn) { /* the bucket's order keys and their places */
    uint4 first[2];
    sel_load(r, r.c0, first);
    sel_chunks<BF16>(r, V, rp.banned, first, [&](const auto &v, int p0, uint32_t ok) {
      float x[EPC];
      sel_scale(v, T, y, te, x);
#pragma unroll
      for (int e = 0; e < EPC; e++)
        if (((ok >> e) & 1u) && sel_rank_bucket(x[e] - M, s) == tb) fn(x[e], p0 + e);
    });
  };
  if (tid == 0) {
    S.lo = ~0u;
    S.hi = 0u;
    S.n = 0u;
  }
  __syncthreads();
  uint32_t lo = ~0u, hi = 0u;
  each([&](float x, int) {
    const uint32_t o = d3s_ordkey(x);
    lo = min(lo, o);
    hi = max(hi, o);
  });
  if (lo <= hi) {
    atomicMin(&S.lo, lo);
    atomicMax(&S.hi, hi);
  }
  __syncthreads();
  lo = S.lo;
  hi = S.hi;
  uint32_t need = (uint32_t)a.k - n; /* of the keys in [lo, hi] */
#pragma unroll 1
  while (lo < hi) {
    const int shift = max(0, 32 - __clz((int)(hi - lo)) - 11);
    static_assert(SEL_NB == 2048 && SEL_NB == 2 * GBLOCK, "11 bits, two counts a thread");
    ((uint2 *)hist)[tid] = make_uint2(0u, 0u);
    __syncthreads();
    each([&](float x, int) {
      const uint32_t o = d3s_ordkey(x);
      if (o >= lo && o <= hi) atomicAdd(&hist[(hi - o) >> shift], 1u);
    });
    __syncthreads();
    const uint2 c = ((const uint2 *)hist)[tid];
    uint32_t all;
    const uint32_t before = block_excl_scan_u32<GNW>(c.x + c.y, sh, all);
    if (before < need && before + c.x + c.y >= need) { /* one thread's */
      const bool second = before + c.x < need;
      S.bin = 2u * tid + (second ? 1u : 0u);
      S.above = before + (second ? c.x : 0u);
      S.count = second ? c.y : c.x;
    }
    __syncthreads();
    need -= S.above;
    hi -= S.bin << shift;
    const uint32_t span = (1u << shift) - 1u;
    lo = hi - lo > span ? hi - span : lo;
    if (S.count == need) { /* every key of [lo, hi]: none is left to choose */
      hi = lo - 1u;
      need = 0u;
    }
    __syncthreads();
  }
  /* (lo == hi: `need` of the equal keys; hi == lo - 1: none) */
  each([&](float x, int i) {
    if (d3s_ordkey(x) > hi) list[atomicAdd(&S.n, 1u)] = composite_key(x, i);
  });
  __syncthreads();
  const int m = (int)S.n;
  int pow2 = 2;
  while (pow2 < m) pow2 <<= 1;
  for (int i = m + tid; i < pow2; i += GBLOCK) list[i] = 0ull; /* sorts last */
  __syncthreads();
  bitonic_sort<GBLOCK>(list, pow2);
  for (int i = tid; i < m; i += GBLOCK) ranked[n + i] = list[i];
  uint32_t base = 0u;
#pragma unroll 1
  for (int t0 = 0; t0 < V && base < need; t0 += TIE * GBLOCK) {
    const int i0 = t0 + TIE * tid;
    uint32_t tie = 0u;
    float tx = 0.0f;
#pragma unroll
    for (int e = 0; e < TIE; e++)
      if (i0 + e < V) {
        const float x = scale_logit(load_logit<BF16>(rowp, i0 + e, rp.banned), T, y, T < __builtin_inff());
        if (d3s_ordkey(x) == lo) {
          tie |= 1u << e;
          tx = x;
        }
      }
    uint32_t all;
    uint32_t at = base + block_excl_scan_u32<GNW>((uint32_t)__popc(tie), sh, all);
#pragma unroll
    for (int e = 0; e < TIE; e++)
      if ((tie >> e) & 1u) {
        if (at < need) ranked[n + m + at] = composite_key(tx, i0 + e);
        at++;
      }
    base += all;
  }
  __syncthreads();
}

/* n composite keys, thread t holding keys t + q GBLOCK of their index order,
 * into list in rank order: a stable radix sort by 8 bits a pass of the order
 * keys' bits that differ (rounded logits: one pass, bf16 ones two), so equal x
 * stay in index order.  Each wave holds a run of the keys and counts its digits
 * alone.  tab: GNW NB words of LDS, sh: two. */
template <int NK>
__device__ __forceinline__ void sel_radix(const uint64_t (&kv)[NK], uint32_t n, uint64_t *list, uint32_t *tab,
                                          uint32_t *sh) {
  static_assert(GNW * NB == 4 * GBLOCK && NB == 4 * WAVE, "a thread clears 16 bytes; a lane sums four digits");
  __shared__ __align__(16) uint32_t dig[NB];
  const int tid = (int)threadIdx.x, lane = lane_id(), wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const uint64_t lt = (1ull << lane) - 1ull;
  if (tid == 0) {
    sh[0] = 0u;
    sh[1] = ~0u;
  }
  __syncthreads();
  uint32_t some = 0u, every = ~0u;
#pragma unroll
  for (int q = 0; q < NK; q++)
    if (tid + q * GBLOCK < (int)n) {
      list[tid + q * GBLOCK] = kv[q];
      some |= (uint32_t)(kv[q] >> 32);
      every &= (uint32_t)(kv[q] >> 32);
    }
  atomicOr(&sh[0], some);
  atomicAnd(&sh[1], every);
  __syncthreads();
  const uint32_t differ = sh[0] & ~sh[1];
  uint32_t *mine = tab + wid * NB;
#pragma unroll 1
  for (int shift = differ ? __builtin_ctz(differ) : 32; shift < 32 && (differ >> shift); shift += 8) {
#pragma unroll
    for (int j = 0; j < 4; j++) tab[tid + j * GBLOCK] = 0u;
    __syncthreads();
    uint64_t key[NK];
    uint32_t at[NK]; /* the key's place among its wave's of that digit */
#pragma unroll
    for (int q = 0; q < NK; q++) {
      const int i = (wid * NK + q) * WAVE + lane;
      const bool in = i < (int)n;
      key[q] = in ? list[i] : 0ull;
      const uint32_t d = (~(uint32_t)(key[q] >> 32) >> shift) & 255u;
      const uint64_t peers = wave_peers<8>(d, __ballot(in));
      const uint32_t below = (uint32_t)__popcll(peers & lt), had = mine[d];
      wave_lds_sync();
      if (in && below == 0u) mine[d] = had + (uint32_t)__popcll(peers);
      wave_lds_sync();
      at[q] = had + below;
      __builtin_amdgcn_sched_barrier(0); /* (one key's ballots at a time: registers) */
    }
    __syncthreads();
    if (tid < NB) { /* each digit's waves in turn */
      uint32_t run = 0u;
#pragma unroll
      for (int w = 0; w < GNW; w++) {
        const uint32_t c = tab[w * NB + tid];
        tab[w * NB + tid] = run;
        run += c;
      }
      dig[tid] = run;
    }
    __syncthreads();
    if (wid == 0) { /* and the digits before: a lane four of them */
      const uint4 c = ((const uint4 *)dig)[lane];
      const uint32_t sum = c.x + c.y + c.z + c.w, before = wave_scan_add_u32(sum) - sum;
      ((uint4 *)dig)[lane] = make_uint4(before, before + c.x, before + c.x + c.y, before + c.x + c.y + c.z);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NK; q++) {
      const uint32_t d = (~(uint32_t)(key[q] >> 32) >> shift) & 255u;
      if ((wid * NK + q) * WAVE + lane < (int)n) list[dig[d] + mine[d] + at[q]] = key[q];
    }
    __syncthreads();
  }
}

/* NQ: k <= NQ GBLOCK */
template <bool BF16, int NQ>
__global__ __launch_bounds__(GBLOCK) void k_sel_sort(SampleArgs a, SelLayout L, int kpow) {
  extern __shared__ uint64_t dyn[];
  uint64_t *sorted = dyn, *bk = dyn + kpow; /* [kpow], [SEL_CAP] */
  __shared__ __align__(16) uint32_t tab[2 * SEL_NB];
  uint32_t *start = tab, *next = tab + SEL_NB;
  __shared__ uint32_t sh[GNW], sbase[SEL_SMAX + 1], many;
  constexpr int PER = SEL_NB / GBLOCK, EPC = BF16 ? 8 : 4, NK = SEL_CAP / GBLOCK;
  static_assert(PER == 2 && SEL_SMAX == WAVE, "");
  const int row = (int)blockIdx.x, tid = (int)threadIdx.x, lane = lane_id();
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  /* everything the first steps need, in one round of loads */
  const SelSeg *sg0 = L.seg + (size_t)row * SEL_SMAX;
  const uint32_t segn = lane < L.nseg ? sg0[lane].count : 0u;
  const uint64_t segs = lane < L.nseg ? sg0[lane].sum : 0ull;
  const uint32_t crowd = sg0[0].crowd;
  const float least = NQ > 1 ? sg0[0].least : 0.0f;
  float u[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int r = tid * NQ + q;
    u[q] = r < a.k ? a.u[(size_t)row * a.k + r] : 0.5f;
  }
  const RowP rp = row_params(a, row);
  const float T = rp.T, y = 1.0f / T;
  float M;
  const SelRow what = sel_row_max(L, row, T, M);
  if (what != SEL_LIVE) { /* a NaN or +inf x: refused; every x -inf: masked */
    write_special(a, row, what == SEL_MASKED);
    return;
  }
  const uint32_t inc = wave_scan_add_u32(segn);
  const uint32_t n = readlane_u(inc, WAVE - 1);
  if (__builtin_expect(__builtin_amdgcn_readfirstlane((int)crowd) != 0, 0)) sel_crowd<BF16>(a, row, rp, M, (int)crowd - 1, n, sorted, bk, start, sh);
  const float lse = M + d3s_logf(d3s_fixsum_to_f32(wave_sum_mod64(segs)));
  /* their buckets: the selection's, or for many keys SEL_NB equal parts of about
   * what they span (any factor ranks them; for few the load and the reciprocal
   * cost more than they save: 8.9 against 9.4 us at k = 30, but [1024, 20000], k =
   * 4096: 165 against 141 us a call) */
  float per = 0.0f;
  if (NQ > 1) {
    const float span = M - least * y;
    per = span > 0.0f ? fminf((float)SEL_NB * __builtin_amdgcn_rcpf(span), 0x1p100f) : 0.0f;
  }
  const float s = sel_rank_scale(T);
  auto place = [&](float x) {
    return NQ > 1 ? (int)fminf((M - x) * per, (float)(SEL_NB - 1)) : sel_rank_bucket(x - M, s);
  };
  next[tid] = 0u;
  next[tid + GBLOCK] = 0u;
  if (tid == 0) many = 0u;
  if (wid == 0) {
    sbase[lane + 1] = inc;
    if (lane == 0) sbase[0] = 0u;
  }
  __syncthreads();
  /* the keys, and how many lie in each bucket */
  const uint64_t *keys = L.keys + (size_t)row * (size_t)L.vstride;
  uint64_t kv[NK];
#pragma unroll
  for (int q = 0; q < NK; q++) {
    const uint32_t i = tid + q * GBLOCK;
    if (i < n) {
      int sg = 0;
#pragma unroll
      for (int step = SEL_SMAX / 2; step >= 1; step >>= 1) sg += sbase[sg + step] <= i ? step : 0;
      kv[q] = keys[(size_t)sg * L.segc * EPC + (i - sbase[sg])];
    }
  }
#pragma unroll
  for (int q = 0; q < NK; q++)
    if (tid + q * GBLOCK < n) {
      const float x = scale_logit(d3s_u2f((uint32_t)(kv[q] >> 32)), T, y, T < __builtin_inff());
      kv[q] = composite_key(x, (int)(uint32_t)kv[q]);
      atomicAdd(&next[place(x)], 1u);
    }
  __syncthreads();
  const uint2 c = ((const uint2 *)next)[tid];
  if (max(c.x, c.y) * ((n + GBLOCK - 1) / GBLOCK) > SEL_PAIRS) many = 1u;
  uint32_t all;
  const uint32_t before = block_excl_scan_u32<GNW>(c.x + c.y, sh, all);
  if (__builtin_expect(__builtin_amdgcn_readfirstlane((int)many) != 0, 0)) { /* (the scan's barriers stand between) */
    sel_radix<NK>(kv, n, bk, tab, sh);
    for (int i = tid; i < min((int)n, a.k); i += GBLOCK) sorted[i] = bk[i];
  } else {
    ((uint2 *)start)[tid] = make_uint2(before, before + c.x);
    ((uint2 *)next)[tid] = make_uint2(before, before + c.x);
    __syncthreads();
    /* the keys by bucket (any order within one) */
#pragma unroll
    for (int q = 0; q < NK; q++)
      if (tid + q * GBLOCK < n) bk[atomicAdd(&next[place(key_x(kv[q]))], 1u)] = kv[q];
    __syncthreads();
    /* next[b] is now bucket b's end; a key's rank: its bucket's start and the
     * larger keys of the bucket */
    for (uint32_t i = tid; i < n; i += GBLOCK) {
      const uint64_t my = bk[i];
      const int b = place(key_x(my));
      const uint32_t e = next[b];
      uint32_t rank = start[b];
      for (uint32_t j = start[b]; j < e; j++) rank += bk[j] > my ? 1u : 0u;
      if (rank < (uint32_t)a.k) sorted[rank] = my;
    }
  }
  __syncthreads();
  sel_tail<NQ>(a, row, lse, rp.top_p, sorted, u);
}

}  // namespace

namespace {

/* dynamic LDS beyond 64 KB must be allowed once per kernel and device (gfx950: 160 KB) */
template <bool BF16, int NQ>
void sort_rows(const SampleArgs &c, const SelLayout &L, hipStream_t s) {
  static std::atomic<bool> done[64];
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 && !done[dev].load(std::memory_order_relaxed) &&
      hipFuncSetAttribute((const void *)k_sel_sort<BF16, NQ>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (SEL_MAX_K + SEL_CAP) * 8) == hipSuccess)
    done[dev].store(true, std::memory_order_relaxed);
  int kpow = 2;
  while (kpow < c.k) kpow <<= 1;
  hipLaunchKernelGGL((k_sel_sort<BF16, NQ>), dim3((unsigned)c.n_rows), dim3(GBLOCK),
                     (size_t)(kpow + SEL_CAP) * sizeof(uint64_t), s, c, L, kpow);
}

template <bool BF16>
void select_rows(const SampleArgs &c, const SelLayout &L, hipStream_t s) {
  const dim3 grid((unsigned)L.nseg, (unsigned)c.n_rows);
  hipLaunchKernelGGL(k_sel_max<BF16>, grid, dim3(SEL_T), 0, s, c, L);
  hipLaunchKernelGGL((k_sel_hist<BF16, false>), grid, dim3(SEL_T), 0, s, c, L);
  hipLaunchKernelGGL((k_sel_gather<BF16, false>), grid, dim3(SEL_T), 0, s, c, L, BkLayout{});
  if (c.k <= GBLOCK)
    sort_rows<BF16, 1>(c, L, s);
  else
    sort_rows<BF16, SEL_MAX_K / GBLOCK>(c, L, s);
}

/* a row's chunks at any start offset */
int64_t sel_nchunks(const SampleArgs &a, int epc) { return ((int64_t)a.vocab + 2 * epc - 2) / epc; }

/* The segments of a row: whole rounds of a workgroup's lanes (SEL_T chunks),
 * as many a segment as leave about SEL_WGS workgroups a launch and at most
 * smax segments a row. */
void sel_segments(SelLayout &L, const SampleArgs &a, Dtype dt, int64_t rows, int smax) {
  const int epc = dt == DT_F32 ? 4 : 8;
  const int64_t rounds = (sel_nchunks(a, epc) + SEL_T - 1) / SEL_T; /* a row's */
  int64_t want = (SEL_WGS + rows - 1) / rows;
  if (want > smax) want = smax;
  int64_t per = rounds / want;
  const int64_t least = (rounds + smax - 1) / smax;
  if (per < least) per = least;
  L.segc = (int)(per * SEL_T);
  L.nseg = (int)((rounds + per - 1) / per);
  L.vstride = rounds * SEL_T * epc;
}

/* one row's workspace: the keys (V and less than a round of 8-element
 * chunks), the segments' tables and records */
size_t sel_row_bytes(const SampleArgs &a, int nseg) {
  const size_t keys = ((size_t)a.vocab + 8u * SEL_T + 16u) * 8u;
  return keys + (size_t)nseg * (SEL_NB + SEL_NG) * 4u + SEL_SMAX * sizeof(SelSeg);
}

}  // namespace

bool sel_takes(const SampleArgs &a) { return a.opgraph && a.k <= SEL_MAX_K && a.vocab > topp_max_vocab(); }

size_t sel_workspace_bytes(const SampleArgs &a, Dtype dt, bool one_row) {
  SelLayout L{};
  sel_segments(L, a, dt, one_row ? 1 : a.n_rows, SEL_SMAX);
  const size_t row = sel_row_bytes(a, L.nseg);
  if (one_row) return row;
  size_t all = row * (size_t)a.n_rows;
  if (all > SEL_WS_CAP) all = SEL_WS_CAP > row ? SEL_WS_CAP : row;
  return all;
}

/* The streaming kernel's time by its measured rows: one row's passes and sort
 * (bf16, k = 100: 37 us at V = 8193, 70 us at 20 000, 436 us at 151 936; fp32
 * a quarter less), and from about 400 rows on their number (1024 rows: 97, 192
 * and 1375 us).  Rather too little than too much. */
double generic_us(const SampleArgs &a, Dtype dt) {
  const double row = 14.0 + (dt == DT_F32 ? 2.0e-3 : 2.7e-3) * a.vocab + 0.01 * a.k;
  const double rounds = 0.62 / 256.0 * a.n_rows;
  return row * (rounds > 1.0 ? rounds : 1.0);
}

bool launch_select(const SampleArgs &a, Dtype dt, void *ws, size_t ws_bytes, hipStream_t s) {
  if (!ws || !sel_takes(a)) return false;
  /* the rows of a launch: as many as ws holds, each launch's rows cut into the
   * segments that suit its number (fewer rows, more segments) */
  int64_t chunk = a.n_rows < 32768 ? a.n_rows : 32768; /* (a grid's second dimension) */
  SelLayout L{};
  for (;; chunk = (chunk + 1) / 2) {
    sel_segments(L, a, dt, chunk, SEL_SMAX);
    if (sel_row_bytes(a, L.nseg) * (size_t)chunk <= ws_bytes) break;
    if (chunk == 1) return false;
  }
  /* (a round of few rows takes 20 to 24 us at any V; 2.7 to 4.5 ps an element) */
  if (!rounds_pay(a, (a.n_rows + chunk - 1) / chunk, 22.0, 4.5e-6, generic_us(a, dt))) return false;
  for (int64_t r0 = 0; r0 < a.n_rows; r0 += chunk) {
    const int64_t n = a.n_rows - r0 < chunk ? a.n_rows - r0 : chunk;
    const SampleArgs c = rows_from(a, dt, r0, n);
    L.keys = (uint64_t *)ws;
    L.seg = (SelSeg *)(L.keys + (size_t)n * (size_t)L.vstride);
    L.cnt = (uint32_t *)(L.seg + (size_t)n * SEL_SMAX); /* (16-byte stores) */
    L.group = L.cnt + (size_t)n * L.nseg * SEL_NB;
    if (dt == DT_F32)
      select_rows<false>(c, L, s);
    else
      select_rows<true>(c, L, s);
  }
  return true;
}

void sel_front_shape(SelLayout &F, const SampleArgs &a, Dtype dt, int64_t rows) {
  sel_segments(F, a, dt, rows, BK_SMAX);
}

size_t sel_front_bytes(const SelLayout &F, bool sums) {
  return (size_t)F.nseg * (sums ? SEL_NB * 12u : (SEL_NB + SEL_NG) * 4u) + SEL_SMAX * sizeof(SelSeg);
}

namespace {
template <bool BF16>
void front(const SampleArgs &a, const BkLayout *L, const SelLayout &F, hipStream_t s) {
  const dim3 grid((unsigned)F.nseg, (unsigned)a.n_rows);
  hipLaunchKernelGGL(k_sel_max<BF16>, grid, dim3(SEL_T), 0, s, a, F);
  if (!L) {
    hipLaunchKernelGGL((k_sel_hist<BF16, true>), grid, dim3(SEL_T), 0, s, a, F);
    return;
  }
  hipLaunchKernelGGL((k_sel_hist<BF16, false>), grid, dim3(SEL_T), 0, s, a, F);
  hipLaunchKernelGGL((k_sel_gather<BF16, true>), grid, dim3(SEL_T), 0, s, a, F, *L);
}
}  // namespace

void launch_select_front(const SampleArgs &a, Dtype dt, const BkLayout *L, const SelLayout &F, hipStream_t s) {
  if (dt == DT_F32)
    front<false>(a, L, F, s);
  else
    front<true>(a, L, F, s);
}

}  // namespace d3s
