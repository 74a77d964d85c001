/* The selecting path: k beyond one wave (65 .. SEL_MAX_K) on rows longer than
 * the nucleus kernel takes, and smaller k on rows wider than the segmented
 * kernel's (gfx950, wave64).  The op graph's order (src/sampling.c:22-49).
 *
 * A row is cut into segments, a workgroup each, so that a few rows fill the
 * chip, and read three times (once from HBM, then from the caches):
 *  k_sel_max: each segment's largest logit (so m = max x, division being
 *     monotone);
 *  k_sel_hist: every x = L / T exactly and its bucket below the max (width
 *     1 / SEL_SCALE, the last one open), counted in LDS and stored per segment
 *     (adding the segments' counts to one table by global atomics took 6.6 us
 *     more, at [32, 151936]); the segment's exact sum of fix40(d3s_expf(x - m));
 *  k_sel_gather: the first bucket at which the row's count reaches k, by groups
 *     of buckets and then within one; the logits that can lie in it or above
 *     (few more than k), each segment's in a region of its own;
 *  k_sel_sort (a workgroup per row): those logits as composite keys, into LDS
 *     by bucket, each key's rank from the larger keys of its own bucket, then
 *     the op graph's tail with lse from the segments' sums.
 * A row with more gathered keys than LDS holds (crowded ties at the k-th
 * element), or whose T is not finite, is sampled by the generic procedure in
 * k_sel_sort's workgroup.  Every result is the oracle's bits.
 *
 * Bound: latency (four launches; k_sel_sort is one workgroup's chain).
 * [32, 151936] bf16, k = 1000: 3.6 + 10.5 + 8.1 + 13.1 us against 438 us for
 * k_generic, one workgroup a row; [1, 8193], k = 65: 20.7 us against 31.3 us;
 * [2048, 32768], k = 4096: 373 us against 776 us. */
#include <atomic>

#include "d3s_rowcore.h"
#include "d3s_select.h"

#pragma clang fp contract(off)

namespace d3s {
namespace {

constexpr int SEL_T = 512; /* threads of a segment's workgroup */
constexpr int SEL_NW = SEL_T / WAVE;
constexpr int SEL_U = 4;   /* 16-byte loads a lane keeps in flight */
constexpr int SEL_CAP = 8192; /* keys k_sel_sort ranks */

/* a wave's run of 16-byte chunks of its segment */
struct SelRun {
  const uint4 *src; /* the row's first chunk */
  int off;          /* elements of it before the row */
  int c0, c1;       /* the wave's chunks [c0, c1) */
};

template <bool BF16>
__device__ __forceinline__ SelRun sel_run(const SampleArgs &a, const SelLayout &L, int row, int seg, int wid) {
  constexpr int ES = BF16 ? 2 : 4, EPC = 16 / ES;
  const char *rowp = (const char *)a.logits + (size_t)row * (size_t)a.row_stride * ES;
  SelRun r;
  r.off = (int)(((uintptr_t)rowp & 15u) / ES);
  r.src = (const uint4 *)(rowp - r.off * ES);
  const int nchunks = (r.off + a.vocab + EPC - 1) / EPC;
  const int wch = (L.segc + SEL_NW - 1) / SEL_NW;
  const int end = min(nchunks, (seg + 1) * L.segc);
  r.c0 = min(end, seg * L.segc + wid * wch);
  r.c1 = min(end, r.c0 + wch);
  return r;
}

/* SEL_U 16-byte loads a lane from chunk `base` of the run on (zeros past it) */
__device__ __forceinline__ void sel_load(const SelRun &r, int base, uint4 (&q)[SEL_U]) {
#pragma unroll
  for (int u = 0; u < SEL_U; u++) {
    const int c = base + u * WAVE + lane_id();
    q[u] = c < r.c1 ? r.src[c] : make_uint4(0u, 0u, 0u, 0u);
  }
}

/* fn(v, p0, ok) for every chunk of the run, `first` the loads of its first
 * SEL_U rows of chunks (issued by the caller ahead of whatever it waits for):
 * v the EPC logits (-inf outside the row and at the banned index), p0 the
 * first one's position, ok the bits of those within the run and the row.
 * Every lane calls fn. */
template <bool BF16, class Fn>
__device__ __forceinline__ void sel_chunks(const SelRun &r, int V, int banned, const uint4 (&first)[SEL_U], Fn &&fn) {
  constexpr int EPC = BF16 ? 8 : 4;
  const int lane = lane_id();
  uint4 q[SEL_U], next[SEL_U];
#pragma unroll
  for (int u = 0; u < SEL_U; u++) q[u] = first[u];
  /* one copy of fn's code: the launch's instruction fetch costs more than the
   * register moves of a rolled loop */
#pragma unroll 1
  for (int base = r.c0; base < r.c1; base += SEL_U * WAVE) {
    sel_load(r, base + SEL_U * WAVE, next);
    const int end = min(r.c1, base + SEL_U * WAVE);
#pragma unroll 1
    for (int cw = base; cw < end; cw += WAVE) { /* cw uniform: the 64 chunks' first */
      const int p0 = (cw + lane) * EPC - r.off, f0 = cw * EPC - r.off;
      const uint32_t w[4] = {q[0].x, q[0].y, q[0].z, q[0].w};
      float v[EPC];
#pragma unroll
      for (int e = 0; e < EPC; e++)
        v[e] = BF16 ? d3s_u2f((e & 1) ? (w[e / 2] & 0xffff0000u) : (w[e / 2] << 16)) : d3s_u2f(w[e]);
      uint32_t ok = (1u << EPC) - 1u;
      if (f0 < 0 || f0 + WAVE * EPC > V || cw + WAVE > r.c1 || (unsigned)(banned - f0) < (unsigned)(WAVE * EPC)) {
        ok = 0u;
#pragma unroll
        for (int e = 0; e < EPC; e++) {
          const bool in = cw + lane < r.c1 && (unsigned)(p0 + e) < (unsigned)V;
          ok |= (in ? 1u : 0u) << e;
          if (!in || p0 + e == banned) v[e] = -__builtin_inff();
        }
      }
      fn(v, p0, ok);
#pragma unroll
      for (int u = 0; u + 1 < SEL_U; u++) q[u] = q[u + 1];
    }
#pragma unroll
    for (int u = 0; u < SEL_U; u++) q[u] = next[u];
  }
}

/* x[e] = v[e] / T for a chunk: the fused division without its range test
 * where every lane's logits allow it (zero divides exactly either way) */
template <int EPC>
__device__ __forceinline__ void sel_scale(const float (&v)[EPC], float T, float y, bool t_easy, float (&x)[EPC]) {
  bool ok = t_easy;
#pragma unroll
  for (int e = 0; e < EPC; e++) {
    const uint32_t ea = (d3s_f2u(v[e]) >> 23) & 0xffu;
    ok = ok && (ea - 67u <= 160u || v[e] == 0.0f);
  }
  if (__all(ok)) {
#pragma unroll
    for (int e = 0; e < EPC; e++) {
      const float q = v[e] * y;
      const float r = __builtin_fmaf(-q, T, v[e]);
      x[e] = __builtin_fmaf(r, y, q);
    }
  } else {
#pragma unroll
    for (int e = 0; e < EPC; e++) x[e] = d3s_div_rn(v[e], T, y);
  }
}

/* what a row's segments' maxima say (every wave alike: lane s reads segment
 * s's): m = max x; false for a row with nothing to gather (refused, all -inf,
 * or T not finite: left to the last kernel) */
__device__ __forceinline__ bool sel_row_max(const SelLayout &L, int row, float T, float &Lmax, float &M) {
  const int lane = lane_id();
  Lmax = wave_maximum_f(lane < L.nseg ? L.seg[(size_t)row * SEL_SMAX + lane].lmax : -__builtin_inff());
  M = 0.0f;
  if (!(T < __builtin_inff()) || d3s_isnan(Lmax) || fabsf(Lmax) == __builtin_inff()) return false;
  M = scale_logit(Lmax, T, 1.0f / T, true);
  return fabsf(M) < __builtin_inff();
}

__device__ __forceinline__ bool sel_t_easy(float T) {
  return ((d3s_f2u(T) >> 23) & 0xffu) - 107u <= 40u; /* d3s_div_rn's range of T */
}

/* the bucket of z = x - m <= 0 (-inf: the last) */
__device__ __forceinline__ int sel_bucket(float z) { return (int)fminf(z * -SEL_SCALE, (float)(SEL_NB - 1)); }

template <bool BF16>
__global__ __launch_bounds__(SEL_T) void k_sel_max(SampleArgs a, SelLayout L) {
  __shared__ float sh[SEL_NW];
  const int seg = (int)blockIdx.x, row = (int)blockIdx.y;
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  const SelRun run = sel_run<BF16>(a, L, row, seg, wid);
  uint4 first[SEL_U];
  sel_load(run, run.c0, first);
  const int banned = a.banned ? a.banned[row] : -1;
  float m = -__builtin_inff();
  sel_chunks<BF16>(run, a.vocab, banned, first, [&](const auto &v, int, uint32_t) {
#pragma unroll
    for (float f : v) m = fmaximum(m, f);
  });
  m = wave_maximum_f(m);
  if (lane_id() == 0) sh[wid] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < SEL_NW; w++) m = fmaximum(m, sh[w]);
    L.seg[(size_t)row * SEL_SMAX + seg].lmax = m;
  }
}

template <bool BF16>
__global__ __launch_bounds__(SEL_T) void k_sel_hist(SampleArgs a, SelLayout L) {
  __shared__ __align__(16) uint32_t cnt[SEL_NB];
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
  float Lmax, M;
  if (!sel_row_max(L, row, T, Lmax, M)) return;
  __syncthreads();
  const bool te = sel_t_easy(T);
  uint64_t acc = 0ull;
  sel_chunks<BF16>(run, a.vocab, rp.banned, first, [&](const auto &v, int, uint32_t ok) {
    constexpr int EPC = BF16 ? 8 : 4;
    float x[EPC];
    sel_scale(v, T, y, te, x);
#pragma unroll
    for (int e = 0; e < EPC; e++) {
      const float z = x[e] - M;
      if ((ok >> e) & 1u) {
        atomicAdd(&cnt[sel_bucket(z)], 1u);
        acc += d3s_fix40_exp(z);
      }
    }
  });
  acc = wave_sum_mod64(acc);
  if (lane_id() == 0) sum[wid] = acc;
  __syncthreads();
  const size_t at = (size_t)row * L.nseg + seg;
  const uint4 c = ((const uint4 *)cnt)[tid];
  ((uint4 *)(L.cnt + at * SEL_NB))[tid] = c;
  uint32_t g = c.x + c.y + c.z + c.w;
  g += dpp_u<0xb1, 0xf>(0u, g);   /* quad_perm [1,0,3,2] */
  g += dpp_u<0x4e, 0xf>(0u, g);   /* quad_perm [2,3,0,1] */
  g += dpp_u<0x141, 0xf>(0u, g);  /* row_half_mirror: the other four of the eight */
  if (tid % (SEL_G / PER) == 0) L.group[at * SEL_NG + tid / (SEL_G / PER)] = g;
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < SEL_NW; w++) acc += sum[w];
    L.seg[(size_t)row * SEL_SMAX + seg].sum = acc;
  }
}

template <bool BF16>
__global__ __launch_bounds__(SEL_T) void k_sel_gather(SampleArgs a, SelLayout L) {
  __shared__ uint32_t part[SEL_NW][SEL_NG], fine[SEL_G], wn[SEL_NW];
  static_assert(SEL_NG == WAVE && SEL_SMAX % SEL_NW == 0, "a lane a group");
  constexpr int EPC = BF16 ? 8 : 4, GL = SEL_SMAX / SEL_NW, FL = SEL_SMAX * SEL_G / SEL_T;
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
  const float T = rp.T;
  float Lmax, M;
  if (!sel_row_max(L, row, T, Lmax, M)) return;
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
    f += s < L.nseg ? L.cnt[(at0 + s) * SEL_NB + tg * SEL_G + tid % SEL_G] : 0u;
  }
  if (f) atomicAdd(&fine[tid % SEL_G], f);
  __syncthreads();
  const uint32_t fin = before + wave_scan_add_u32(lane < SEL_G ? fine[lane] : 0u);
  const int tb = tg * SEL_G + (int)__builtin_ctzll(__ballot(fin >= k) | (1ull << (SEL_G - 1)));
  /* every logit of the buckets up to tb reaches Lc: (tb + 1) / SEL_SCALE below
   * m, with room for the roundings of x, of x - m and of this bound (a few
   * elements below them may as well: the set holds every element above any of
   * its own, which is all that k_sel_sort asks) */
  float Lc = -__builtin_inff();
  if (tb < SEL_NB - 1) {
    const float xc = M - ((float)(tb + 1) * (1.0f / SEL_SCALE)) * 1.0001f;
    Lc = (xc - (fabsf(M) + fabsf(xc) + 1.0f) * 0x1p-20f) * T;
    Lc = Lc - fabsf(Lc) * 0x1p-20f;
    if (!(Lc >= -0x1.fffffep127f)) Lc = -__builtin_inff();
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
  if (tid == 0) L.seg[(size_t)row * SEL_SMAX + seg].count = tot;
  if (n == 0u) return;
  uint64_t *out = L.keys + (size_t)row * (size_t)L.vstride + (size_t)seg * L.segc * EPC;
  sel_chunks<BF16>(run, a.vocab, rp.banned, first, [&](const auto &v, int p0, uint32_t ok) {
    const uint32_t m = pick(v, ok);
    if (__ballot(m != 0u) == 0ull) return;
    const uint32_t c = (uint32_t)__popc(m);
    const uint32_t inc = wave_scan_add_u32(c);
    uint32_t slot = at + inc - c;
#pragma unroll
    for (int e = 0; e < EPC; e++)
      if ((m >> e) & 1u) out[slot++] = ((uint64_t)d3s_f2u(v[e]) << 32) | (uint32_t)(p0 + e);
    at += readlane_u(inc, 63);
  });
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

/* NQ: k <= NQ GBLOCK */
template <bool BF16, int NQ>
__global__ __launch_bounds__(GBLOCK) void k_sel_sort(SampleArgs a, SelLayout L, int kpow) {
  extern __shared__ uint64_t dyn[];
  uint64_t *sorted = dyn, *bk = dyn + kpow; /* [kpow], [SEL_CAP] */
  __shared__ uint32_t start[SEL_NB], next[SEL_NB];
  __shared__ uint32_t sh[GNW], sbase[SEL_SMAX + 1];
  constexpr int PER = SEL_NB / GBLOCK, EPC = BF16 ? 8 : 4, NK = SEL_CAP / GBLOCK;
  static_assert(PER == 2 && SEL_SMAX == WAVE, "");
  const int row = (int)blockIdx.x, tid = (int)threadIdx.x, lane = lane_id();
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  /* everything the first steps need, in one round of loads */
  const SelSeg *sg0 = L.seg + (size_t)row * SEL_SMAX;
  const uint32_t segn = lane < L.nseg ? sg0[lane].count : 0u;
  const uint64_t segs = lane < L.nseg ? sg0[lane].sum : 0ull;
  float u[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int r = tid * NQ + q;
    u[q] = r < a.k ? a.u[(size_t)row * a.k + r] : 0.5f;
  }
  const RowP rp = row_params(a, row);
  const float T = rp.T, y = 1.0f / T;
  float Lmax, M;
  const bool live = sel_row_max(L, row, T, Lmax, M);
  const uint32_t inc = wave_scan_add_u32(segn);
  const uint32_t n = live ? readlane_u(inc, WAVE - 1) : 0u;
  /* T not finite, or a crowded last bucket */
  const bool generic = live ? n > (uint32_t)SEL_CAP : !(T < __builtin_inff());
  if (generic) {
    generic_row<BF16>(a, row, kpow, dyn);
    return;
  }
  if (!live) { /* a NaN or +inf x: refused; every x -inf: masked */
    write_special(a, row, Lmax == -__builtin_inff() || M == -__builtin_inff());
    return;
  }
  const float lse = M + d3s_logf(d3s_fixsum_to_f32(wave_sum_mod64(segs)));
  next[tid] = 0u;
  next[tid + GBLOCK] = 0u;
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
      const float x = scale_logit(d3s_u2f((uint32_t)(kv[q] >> 32)), T, y, true);
      kv[q] = composite_key(x, (int)(uint32_t)kv[q]);
      atomicAdd(&next[sel_bucket(x - M)], 1u);
    }
  __syncthreads();
  const uint2 c = ((const uint2 *)next)[tid];
  uint32_t all;
  const uint32_t before = block_excl_scan_u32<GNW>(c.x + c.y, sh, all);
  ((uint2 *)start)[tid] = make_uint2(before, before + c.x);
  ((uint2 *)next)[tid] = make_uint2(before, before + c.x);
  __syncthreads();
  /* the keys by bucket (any order within one) */
#pragma unroll
  for (int q = 0; q < NK; q++)
    if (tid + q * GBLOCK < n) bk[atomicAdd(&next[sel_bucket(key_x(kv[q]) - M)], 1u)] = kv[q];
  __syncthreads();
  /* next[b] is now bucket b's end; a key's rank: its bucket's start and the
   * larger keys of the bucket */
  for (uint32_t i = tid; i < n; i += GBLOCK) {
    const uint64_t my = bk[i];
    const int b = sel_bucket(key_x(my) - M);
    const uint32_t e = next[b];
    uint32_t rank = start[b];
    for (uint32_t j = start[b]; j < e; j++) rank += bk[j] > my ? 1u : 0u;
    if (rank < (uint32_t)a.k) sorted[rank] = my;
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
  hipLaunchKernelGGL(k_sel_hist<BF16>, grid, dim3(SEL_T), 0, s, c, L);
  hipLaunchKernelGGL(k_sel_gather<BF16>, grid, dim3(SEL_T), 0, s, c, L);
  if (c.k <= GBLOCK)
    sort_rows<BF16, 1>(c, L, s);
  else
    sort_rows<BF16, SEL_MAX_K / GBLOCK>(c, L, s);
}

/* a row's chunks at any start offset */
int64_t sel_nchunks(const SampleArgs &a, int epc) { return ((int64_t)a.vocab + 2 * epc - 2) / epc; }

/* The segments of a row: whole rounds of a workgroup's lanes (SEL_T chunks),
 * as many a segment as leave about SEL_WGS workgroups a launch and at most
 * SEL_SMAX segments a row. */
void sel_segments(SelLayout &L, const SampleArgs &a, Dtype dt, int64_t rows) {
  const int epc = dt == DT_F32 ? 4 : 8;
  const int64_t rounds = (sel_nchunks(a, epc) + SEL_T - 1) / SEL_T; /* a row's */
  int64_t want = (SEL_WGS + rows - 1) / rows;
  if (want > SEL_SMAX) want = SEL_SMAX;
  int64_t per = rounds / want;
  const int64_t least = (rounds + SEL_SMAX - 1) / SEL_SMAX;
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
  sel_segments(L, a, dt, one_row ? 1 : a.n_rows);
  const size_t row = sel_row_bytes(a, L.nseg);
  if (one_row) return row;
  size_t all = row * (size_t)a.n_rows;
  if (all > SEL_WS_CAP) all = SEL_WS_CAP > row ? SEL_WS_CAP : row;
  return all;
}

bool launch_select(const SampleArgs &a, Dtype dt, void *ws, size_t ws_bytes, hipStream_t s) {
  if (!ws || !sel_takes(a)) return false;
  /* the rows of a launch: as many as ws holds, each launch's rows cut into the
   * segments that suit its number (fewer rows, more segments) */
  int64_t chunk = a.n_rows < 32768 ? a.n_rows : 32768; /* (a grid's second dimension) */
  SelLayout L{};
  for (;; chunk = (chunk + 1) / 2) {
    sel_segments(L, a, dt, chunk);
    if (sel_row_bytes(a, L.nseg) * (size_t)chunk <= ws_bytes) break;
    if (chunk == 1) return false;
  }
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

}  // namespace d3s
