/* The selecting path's row layout in the workspace (d3s_select.hip), and the
 * sorting path's (d3s_bigk.hip), whose keys its kernels can gather. */
#ifndef D3S_SELECT_H
#define D3S_SELECT_H

#include "d3s_rowcore.h"

#pragma clang fp contract(off)

namespace d3s {
namespace {

constexpr int SEL_SMAX = 64;         /* segments per row (at most) */
constexpr int SEL_WGS = 512;         /* workgroups a launch aims at: two per CU */
constexpr int SEL_NB = 2048;         /* buckets below a row's max */
constexpr float SEL_SCALE = 64.0f;   /* buckets per unit of x: 32 units, where the terms of the
                                        exact sum end (e^-28 < 2^-40) */
constexpr float SEL_NEAR = 2.0f;     /* the selection's buckets: this, plus the distance, by its */
constexpr int SEL_OCT_LOG2 = 8;      /* exponent and 8 mantissa bits: 8 octaves of 256 */
constexpr int SEL_G = 32;            /* buckets a group */
constexpr int SEL_NG = SEL_NB / SEL_G;
constexpr int SEL_MAX_K = 4096;      /* largest k k_sel_sort takes */
constexpr int BK_SMAX = 16;          /* the sorting path's segments per row (at most) */
constexpr size_t SEL_WS_CAP = (size_t)256 << 20; /* workspace of one launch (then fewer rows) */

}  // namespace

struct SelSeg {
  float lmax;     /* the segment's largest logit (NaN propagates) */
  uint32_t count; /* its keys gathered */
  uint32_t masked; /* some logit is -inf (asked for at T = +inf only) */
  uint32_t crowd;  /* the row's bucket (+ 1) whose elements are not gathered, being too many; else 0 */
  float least;     /* what the row's gathered logits reach */
  uint64_t sum;   /* its exact sum of fix40(d3s_expf(x - m)) */
};

struct SelLayout {
  uint64_t *keys;  /* [n][vstride]: segment s's at s segc EPC: (logit bits, index) */
  uint32_t *cnt;   /* [n][nseg][SEL_NB]: the segment's elements of each bucket (0 for the last) */
  uint32_t *group; /* [n][nseg][SEL_NG]: and of each group of buckets */
  uint64_t *csum;  /* [n][nseg][SEL_NB]: the buckets' exact sums (for the wide nucleus path) */
  SelSeg *seg;     /* [n][SEL_SMAX] */
  int64_t vstride;
  int nseg, segc;  /* segments per row, 16-byte chunks per segment */
};

/* a segment's record: the row's max and its refusal flag, the segment's exact
 * sum (k_sel_gather's, or k_bk_keys' max and the row's first pass's sum), its
 * keys and their digits; then, for the segment's ranks after the sort, the sums
 * of their terms fix40(d3s_expf(x_r - lse)) and fix40(d3s_expf(x_r - x_0))
 * (k_bk_sums) and their race's first maximum (k_bk_race); segment 0's record
 * also holds the row's cut and 1 / kept sum (k_bk_cut) */
struct __align__(16) BkMeta {
  float max;
  uint32_t flags; /* bit 0: refused */
  uint64_t sum;
  uint32_t kor, kand; /* OR and AND of the segment's digit words */
  uint32_t klow;      /* OR of the low 16 bits of its x */
  uint32_t count;     /* its keys */
  uint64_t psum, ksum;
  float best;
  int bestr;
  int cut;
  float inv;
};

/* a launch's rows in the workspace (the tile sums after the records): the rows' key buffers, their count
 * tables ([row][pass][segment][digit]: filled by the pass before each), the
 * segments' counts of digits 0 and 2 in index order ([row][2][segment][digit]:
 * the first pass's), then their segments' records */
struct BkLayout {
  uint64_t *keys; /* [n][2][vstride]; before the first pass segment s's at s rstride of the first */
  uint32_t *hist; /* [n][4][BK_SMAX][NB] */
  uint32_t *hidx; /* [n][2][BK_SMAX][NB] */
  BkMeta *meta;   /* [n][BK_SMAX] */
  uint64_t *tsum; /* [n][ntiles][2]: each tile's exact prefix and kept-sum terms' sums (k_bk_sums) */
  int ntiles;     /* tiles of BK_T ranks a row */
  int64_t vstride;
  int nseg;       /* segments per row */
  int rstride;
  int pass0;      /* the first pass launched: 2 when every row's x is known to
                     have zero low 16 bits (bf16 logits at a scalar T of 1),
                     else 0 */
  bool summed;    /* the exact sums are in the records before the first pass */
};

namespace {

/* the sort digit of a composite key in a pass: byte `pass` of ~ordkey(x)
 * (ascending ~ordkey is descending x) */
__device__ __forceinline__ uint32_t bk_digit(uint64_t key, int pass) {
  return (uint32_t)((~key) >> (32 + 8 * pass)) & 0xffu;
}

/* the wave's lanes whose d has the same low `bits` bits as this lane's
 * (among the lanes in `live`), by one ballot per bit */
template <int BITS>
__device__ __forceinline__ uint64_t wave_peers(uint32_t d, uint64_t live) {
  uint64_t peers = live;
#pragma unroll
  for (int b = 0; b < BITS; b++) {
    const uint64_t bb = __ballot((d >> b) & 1u);
    peers &= ((d >> b) & 1u) ? bb : ~bb;
  }
  return peers;
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int l) {
  return ((uint64_t)readlane_u((uint32_t)(v >> 32), l) << 32) | readlane_u((uint32_t)v, l);
}

constexpr int SEL_T = 512; /* threads of a segment's workgroup */
constexpr int SEL_NW = SEL_T / WAVE;
constexpr int SEL_U = 4;   /* 16-byte loads a lane keeps in flight */

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

/* U 16-byte loads a lane from chunk `base` of the run on (zeros past it) */
template <int U>
__device__ __forceinline__ void sel_load(const SelRun &r, int base, uint4 (&q)[U]) {
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int c = base + u * WAVE + lane_id();
    q[u] = c < r.c1 ? r.src[c] : make_uint4(0u, 0u, 0u, 0u);
  }
}

/* fn(v, p0, ok) for every chunk of the run, `first` the loads of its first
 * U rows of chunks (issued by the caller ahead of whatever it waits for):
 * v the EPC logits (-inf outside the row and at the banned index), p0 the
 * first one's position, ok the bits of those within the run and the row.
 * Every lane calls fn. */
template <bool BF16, int U, class Fn>
__device__ __forceinline__ void sel_chunks(const SelRun &r, int V, int banned, const uint4 (&first)[U], Fn &&fn) {
  constexpr int EPC = BF16 ? 8 : 4;
  const int lane = lane_id();
  uint4 q[U], next[U];
#pragma unroll
  for (int u = 0; u < U; u++) q[u] = first[u];
  /* one copy of fn's code: the launch's instruction fetch costs more than the
   * register moves of a rolled loop */
#pragma unroll 1
  for (int base = r.c0; base < r.c1; base += U * WAVE) {
    sel_load(r, base + U * WAVE, next);
    const int end = min(r.c1, base + U * WAVE);
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
      for (int u = 0; u + 1 < U; u++) q[u] = q[u + 1];
    }
#pragma unroll
    for (int u = 0; u < U; u++) q[u] = next[u];
  }
}

/* x[e] = v[e] / T for a chunk: the fused division without its range test
 * where every lane's logits allow it (zero divides exactly either way) */
template <int EPC>
__device__ __forceinline__ void sel_scale(const float (&v)[EPC], float T, float y, bool t_easy, float (&x)[EPC]) {
  if (T == 1.0f) { /* (uniform) */
#pragma unroll
    for (int e = 0; e < EPC; e++) x[e] = v[e];
    return;
  }
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
    for (int e = 0; e < EPC; e++) x[e] = scale_logit(v[e], T, y, T < __builtin_inff());
  }
}

/* what a row's segments' maxima say (every wave alike: lane s reads segment
 * s's) */
enum SelRow { SEL_LIVE, SEL_REFUSED, SEL_MASKED };
__device__ __forceinline__ SelRow sel_row_max(const SelLayout &L, int row, float T, float &M) {
  const int lane = lane_id();
  const SelSeg *sg = L.seg + (size_t)row * SEL_SMAX;
  const float Lmax = wave_maximum_f(lane < L.nseg ? sg[lane].lmax : -__builtin_inff());
  M = 0.0f;
  if (d3s_isnan(Lmax) || Lmax == __builtin_inff() || d3s_isnan(T)) return SEL_REFUSED;
  if (!(T < __builtin_inff())) /* x = L / +inf: zero, or NaN when some L is -inf */
    return __ballot(lane < L.nseg && sg[lane].masked != 0u) ? SEL_REFUSED : SEL_LIVE;
  if (Lmax == -__builtin_inff()) return SEL_MASKED;
  M = scale_logit(Lmax, T, 1.0f / T, true);
  return M == __builtin_inff() ? SEL_REFUSED : M == -__builtin_inff() ? SEL_MASKED : SEL_LIVE;
}

__device__ __forceinline__ bool sel_t_easy(float T) {
  return ((d3s_f2u(T) >> 23) & 0xffu) - 107u <= 40u; /* d3s_div_rn's range of T */
}

/* the bucket of z = x - m <= 0 (-inf: the last) */
__device__ __forceinline__ int sel_bucket(float z) { return (int)fminf(z * -SEL_SCALE, (float)(SEL_NB - 1)); }

/* a bound every logit of x >= xc - (the roundings of x, of x - m and of this
 * bound) reaches */
__device__ __forceinline__ float sel_logit_from(float M, float T, float xc) {
  const float ninf = -__builtin_inff();
  float Lc = (xc - (fabsf(M) + fabsf(xc) + 1.0f) * 0x1p-20f) * T;
  Lc = Lc - fabsf(Lc) * 0x1p-20f;
  return Lc >= -0x1.fffffep127f ? Lc : ninf;
}

/* a bound every logit of the buckets up to b reaches: (b + 1) / SEL_SCALE below
 * m */
__device__ __forceinline__ float sel_logit_bound(float M, float T, int b) {
  if (b >= SEL_NB - 1 || !(T < __builtin_inff())) return -__builtin_inff();
  return sel_logit_from(M, T, M - ((float)(b + 1) * (1.0f / SEL_SCALE)) * 1.0001f);
}

/* The selection's buckets, of z times s = sel_rank_scale(T): what they divide
 * is a row's logits, since the k-th of a model's logits lies at some 8 to 15
 * units of L below the first at any T (x = L / T: 0.5 to 1.5 million at the
 * smallest T, where buckets of x held nearly all of a row in the last).  1/128
 * wide in the first 2 units, 1/32 from 6 to 14, and so on to 510 units: rows of
 * other scales keep a relative width of 1/256.  (Equal widths and then 32 an octave,
 * four instructions an element more: 540 us against 490 us at [256, 700001].) */
__device__ __forceinline__ float sel_rank_scale(float T) { return fminf(T, 1.0f); }

/* z <= 0 */
__device__ __forceinline__ int sel_rank_bucket(float z, float s) {
  constexpr uint32_t near = __builtin_bit_cast(uint32_t, SEL_NEAR) >> (23 - SEL_OCT_LOG2);
  const uint32_t t = d3s_f2u(__builtin_fmaf(z, -s, SEL_NEAR)) >> (23 - SEL_OCT_LOG2);
  return (int)(min(t, near + (uint32_t)SEL_NB - 1u) - near);
}

/* the distance (times s) at which bucket b ends */
__device__ __forceinline__ float sel_rank_end(int b) {
  return d3s_u2f((uint32_t)(b + 1 + (int)(__builtin_bit_cast(uint32_t, SEL_NEAR) >> (23 - SEL_OCT_LOG2)))
                 << (23 - SEL_OCT_LOG2)) - SEL_NEAR;
}

/* sel_logit_bound for them (y = 1 / T) */
__device__ __forceinline__ float sel_rank_bound(float M, float T, float y, int b) {
  if (b >= SEL_NB - 1 || !(T < __builtin_inff())) return -__builtin_inff();
  return sel_logit_from(M, T, M - sel_rank_end(b) * fmaxf(y, 1.0f) * 1.0001f);
}

/* the least logit of the buckets up to b (+inf: none), over the order keys, 64
 * of them at a time: x, x - m and its bucket are monotone in the logit.  Every
 * lane of the wave calls it. */
__device__ __forceinline__ float sel_rank_least(float M, float T, float y, float s, int b) {
  uint32_t lo = d3s_ordkey(-__builtin_inff()), hi = d3s_ordkey(__builtin_inff()); /* lo: not; hi: is */
#pragma unroll 1
  while (hi - lo > 1u) {
    const uint32_t step = (hi - lo + 63u) / 64u, at = min(hi, lo + (uint32_t)lane_id() * step);
    const float x = scale_logit(d3s_from_ordkey(at), T, y, T < __builtin_inff());
    /* (past the row's max: in the first bucket) */
    const bool is = at == hi || (at > lo && sel_rank_bucket(fminf(x - M, 0.0f), s) <= b);
    const uint64_t m = __ballot(is);
    const int l = m ? (int)__builtin_ctzll(m) : WAVE; /* (lane 0 is at lo) */
    const uint32_t first = l < WAVE ? min(hi, lo + (uint32_t)l * step) : hi;
    lo = lo + (uint32_t)(l - 1) * step;
    hi = first;
  }
  return d3s_from_ordkey(hi);
}

}  // namespace

/* rows [r0, r0 + n) of a call */
inline SampleArgs rows_from(const SampleArgs &a, Dtype dt, int64_t r0, int64_t n) {
  SampleArgs c = a;
  c.n_rows = (int)n;
  c.logits = (const char *)a.logits + (size_t)r0 * (size_t)a.row_stride * (dt == DT_F32 ? 4 : 2);
  c.u = a.u + (size_t)r0 * a.k;
  if (a.temperature) c.temperature = a.temperature + r0;
  if (a.top_p) c.top_p = a.top_p + r0;
  if (a.banned) c.banned = a.banned + r0;
  c.ids = a.ids + r0;
  if (a.probs) c.probs = a.probs + (size_t)r0 * a.k;
  if (a.cand) c.cand = a.cand + (size_t)r0 * a.k;
  return c;
}

/* Whether rows taken in `groups` rounds of launches, for want of workspace, are
 * worth it against one launch of the streaming kernel: a round's latency
 * (group_us) and the elements' work (element_us) against generic_us.  One round
 * always is.  [1024, 20000] bf16, k = 100: 512 rounds of two rows took 20.4 ms, 64
 * of 16 rows 1.36 ms, the streaming kernel 0.19 ms, one round 0.076 ms. */
double generic_us(const SampleArgs &a, Dtype dt);
inline bool rounds_pay(const SampleArgs &a, int64_t groups, double group_us, double element_us, double other_us) {
  return groups <= 1 || (double)groups * group_us + element_us * (double)a.n_rows * (double)a.vocab <= other_us;
}

/* The selecting kernels as a front: with L, the sorting path's (k < V: only the
 * elements that can rank below k, as keys in L; fills its records and counts);
 * without, the wide nucleus path's (each segment's counts and exact sums per
 * bucket). */
void launch_select_front(const SampleArgs &a, Dtype dt, const BkLayout *L, const SelLayout &F, hipStream_t s);
/* the front's segments (F.nseg, F.segc, F.vstride) for launches of `rows` rows,
 * and its workspace for one row */
void sel_front_shape(SelLayout &F, const SampleArgs &a, Dtype dt, int64_t rows);
size_t sel_front_bytes(const SelLayout &F, bool sums);

}  // namespace d3s

#endif
