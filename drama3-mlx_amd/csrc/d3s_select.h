/* The selecting path's row layout in the workspace (d3s_select.hip). */
#ifndef D3S_SELECT_H
#define D3S_SELECT_H

#include "d3s_device.h"

namespace d3s {
namespace {

constexpr int SEL_SMAX = 64;         /* segments per row (at most) */
constexpr int SEL_WGS = 512;         /* workgroups a launch aims at: two per CU */
constexpr int SEL_NB = 2048;         /* buckets below a row's max */
constexpr float SEL_SCALE = 64.0f;   /* buckets per unit of x: 32 units, where the terms of the
                                        exact sum end (e^-28 < 2^-40) */
constexpr int SEL_MAX_K = 4096;      /* largest k k_sel_sort takes */
constexpr size_t SEL_WS_CAP = (size_t)256 << 20; /* workspace of one launch (then fewer rows) */

struct SelSeg {
  float lmax;     /* the segment's largest logit (NaN propagates) */
  uint32_t count; /* its keys gathered */
  uint64_t sum;   /* its exact sum of fix40(d3s_expf(x - m)) */
};

constexpr int SEL_G = 32;                /* buckets a group */
constexpr int SEL_NG = SEL_NB / SEL_G;   /* groups */

struct SelLayout {
  uint64_t *keys;  /* [n][vstride]: segment s's at s segc EPC: (logit bits, index) */
  uint32_t *cnt;   /* [n][nseg][SEL_NB]: the segment's elements of each bucket */
  uint32_t *group; /* [n][nseg][SEL_NG]: and of each group of buckets */
  SelSeg *seg;     /* [n][SEL_SMAX] */
  int64_t vstride;
  int nseg, segc;  /* segments per row, 16-byte chunks per segment */
};

/* sum over the wave of per-lane 64-bit values, exact modulo 2^64 (three
 * 24-bit parts, each summed in 32 bits) */
__device__ __forceinline__ uint64_t wave_sum_mod64(uint64_t v) {
  const uint32_t p0 = wave_sum_u32((uint32_t)(v & 0xffffffu));
  const uint32_t p1 = wave_sum_u32((uint32_t)((v >> 24) & 0xffffffu));
  const uint32_t p2 = wave_sum_u32((uint32_t)(v >> 48));
  return (uint64_t)p0 + ((uint64_t)p1 << 24) + ((uint64_t)p2 << 48);
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

}  // namespace d3s

#endif
