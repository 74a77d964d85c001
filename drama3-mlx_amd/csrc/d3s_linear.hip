/* k_linear_rows: the heads' logits for several hidden rows at once (gfx950,
 * wave64), in the reference's single-row gemv order (src/mlxu.c:365-400),
 * bit for bit, on the matrix cores.
 *
 * The order makes each logit 32 independent chains (lane l of the gemv adds
 * the products of elements c*128 + 4l + t over the blocks c in order, each
 * step one fused multiply-add in fp32) and a tree over the chains.  A K = 1
 * fp32 MFMA is exactly one such step for a whole tile: v_mfma_f32_16x16x1_4b
 * adds one product to each of 4 x 16 x 16 accumulators with one rounding
 * (measured equal to v_fma_f32 on random, subnormal, overflowing and
 * arbitrary bit patterns; a NaN stays a NaN).  So the four "blocks" of the
 * instruction are four chains of one 16 (weight rows) x 16 (hidden rows) tile
 * of logits, and the instructions of a chain run in the gemv's element order.
 *
 * A workgroup takes MT x NT tiles, its waves sharing the 32 chains (four or
 * eight each), so one fragment of weights and one of hidden rows feed each
 * MFMA from LDS.  The rows are staged through LDS a few 128-element blocks at a
 * time in whole 256-byte lines (lanes reading their own chains' pieces of 16
 * rows straight from memory: no faster, and slower the more loads in flight,
 * every 128-byte line being shared by two waves).  After the last block the
 * chains meet in LDS: a thread sums an output's 32 partial sums in the gemv's
 * tree.  Rows past the last read as zeros and are not stored.
 *
 * Bound: fp32 matrix issue.  A 16x16x1_4b takes 32 cycles for 1024 products
 * (65 T products a second measured) and the operands' bf16 to fp32 shifts do
 * not hide behind it.  [64, 2048] x [4097, 2048]: 15.5 us against 138.7 us for
 * k_linear's row after row (8.3 us of MFMA alone); 16 rows 7.7 us against
 * 37.1 us, 256 rows 46.5 us against 546 us (33 us of MFMA alone). */
#include "d3s_gemv.h"

#pragma clang fp contract(off)

namespace d3s {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int LR_TILE = 16; /* weight rows and hidden rows of a tile */
constexpr int LR_XCDS = 8;  /* workgroups go to the XCDs in turn */
/* V's remainder past whole weight tiles, up to this many logits a row, is
 * taken a half-wave a logit (gemv_half_wave) by workgroups after the tiles':
 * V = 4097 at 64 rows is 256 tiles of 32 x 32, one a CU, where a 257th
 * column of tiles would double the launch (16.4 us against 19.0 us with 16 x
 * 16 tiles, five a CU on some CUs instead of four) */
constexpr int LR_REM = 4;

/* MT, NT: tiles of weight rows and of hidden rows a workgroup takes; H:
 * accumulator tiles (of four chains) a wave holds per pair of them, so 8 / H
 * waves a workgroup; CB: 128-element blocks a stage holds. */
template <int MT, int NT, int H, int CB, int MINW>
__global__ __launch_bounds__(WAVE * 8 / H, MINW) void k_linear_rows(const uint16_t *x, const uint16_t *w, int K,
                                                                    int V, int n_rows, int ntiles, int vmain,
                                                                    uint16_t *y) {
  constexpr int T = WAVE * 8 / H;
  constexpr int ROWS = LR_TILE * (MT + NT); /* rows of a stage: weights, then hidden rows */
  constexpr int STAGE = ROWS * CB * 16;     /* 16-byte chunks of a stage */
  constexpr int NL = STAGE / T;             /* 16-byte loads a thread makes per stage */
  constexpr int RJ = T / (16 * CB);         /* rows a workgroup's load covers */
  static_assert(LR_TILE * MT % RJ == 0, "a load is of weights or of hidden rows");
  constexpr int PH = T / 256;               /* tiles of logits summed at once */
  constexpr int RED = PH * 32 * 64;         /* 16-byte chunks of their partial sums */
  __shared__ uint4 lds[2 * STAGE > RED ? 2 * STAGE : RED];
  const int tid = (int)threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = lane_id(), i = lane & 15, b = lane >> 4;
  /* the hidden-row tiles of one weight tile run one after the other on one
   * XCD: its L2 serves the weights to all but the first */
  const int per_x = (vmain + LR_XCDS * LR_TILE * MT - 1) / (LR_XCDS * LR_TILE * MT) * ntiles;
  if ((int)blockIdx.x >= per_x * LR_XCDS) { /* the logits past vmain, one a half-wave */
    const LinearArgs la{x, w, K, V, n_rows, y};
    const int o = (((int)blockIdx.x - per_x * LR_XCDS) * (T / WAVE) + wid) * 2 + (lane >> 5);
    const int rem = V - vmain, n = min(o / rem, n_rows - 1), r = vmain + o % rem;
    const float sum = gemv_half_wave(la, n, r, lane & 31);
    if ((lane & 31) == 0 && o < rem * n_rows) y[(size_t)n * V + r] = d3s_f32_to_bf16_rn(sum);
    return;
  }
  const int xcd = (int)blockIdx.x % LR_XCDS, s = (int)blockIdx.x / LR_XCDS;
  const int n0 = (s % ntiles) * LR_TILE * NT, v0 = ((s / ntiles) * LR_XCDS + xcd) * LR_TILE * MT;
  if (v0 >= vmain) return;
  const int KB = K / 128, NS = (KB + CB - 1) / CB;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(w + (size_t)v0 * K), (short)0, min(V - v0, LR_TILE * MT) * K * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(x + (size_t)n0 * K), (short)0, min(n_rows - n0, LR_TILE * NT) * K * 2, 0x00020000);

  /* load j of a stage: chunk `ch` of block `cb` of row j * RJ + lr */
  const int ch = tid & 15, cb = (tid >> 4) % CB, lr = tid / (16 * CB);
  const int at = lr * K * 2 + cb * 256 + ch * 16;
  u32x4 st[NL];
  auto load = [&](int stage) {
    const int so = min(stage, NS - 1) * CB * 256;
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int row = j * RJ; /* (+ lr) */
      st[j] = row < LR_TILE * MT ? __builtin_amdgcn_raw_buffer_load_b128(wr, at + row * K * 2, so, 0)
                                 : __builtin_amdgcn_raw_buffer_load_b128(xr, at + (row - LR_TILE * MT) * K * 2, so, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  /* a row's 16 chunks of a block are stored at chunk ^ (row % 16): the 16
   * rows a wave reads one chunk of lie in 16 different bank groups */
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int row = j * RJ + lr;
      lds[buf * STAGE + (row * CB + cb) * 16 + (ch ^ (row & 15))] = make_uint4(st[j][0], st[j][1], st[j][2], st[j][3]);
    }
  };

  f32x16 acc[MT][NT][H];
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int m = 0; m < NT; m++)
#pragma unroll
      for (int h = 0; h < H; h++)
#pragma unroll
        for (int j = 0; j < 16; j++) acc[a][m][h][j] = 0.0f;
  const int rd = (H == 2 ? 4 * wid + b : 2 * wid + (b >> 1)) ^ i; /* this lane's chunk of a row */
  auto frag = [&](uint32_t (&q)[2 * H], int buf, int row, int c) {
    const uint4 *p = &lds[buf * STAGE + (row * CB + c) * 16 + rd];
    if constexpr (H == 2) {
      const uint4 v = *p;
      q[0] = v.x, q[1] = v.y, q[2] = v.z, q[3] = v.w;
    } else {
      const uint2 v = ((const uint2 *)p)[b & 1];
      q[0] = v.x, q[1] = v.y;
    }
  };
  auto step1 = [&](int buf, int c) {
    uint32_t wq[MT][2 * H], xq[NT][2 * H];
#pragma unroll
    for (int a = 0; a < MT; a++) frag(wq[a], buf, LR_TILE * a + i, c);
#pragma unroll
    for (int m = 0; m < NT; m++) frag(xq[m], buf, LR_TILE * (MT + m) + i, c);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int h = 0; h < H; h++) {
        float wf[MT], xf[NT];
#pragma unroll
        for (int a = 0; a < MT; a++) {
          const uint32_t u = wq[a][2 * h + t / 2];
          wf[a] = d3s_u2f(t & 1 ? u & 0xffff0000u : u << 16);
        }
#pragma unroll
        for (int m = 0; m < NT; m++) {
          const uint32_t u = xq[m][2 * h + t / 2];
          xf[m] = d3s_u2f(t & 1 ? u & 0xffff0000u : u << 16);
        }
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
          for (int m = 0; m < NT; m++)
            acc[a][m][h] = __builtin_amdgcn_mfma_f32_16x16x1f32(wf[a], xf[m], acc[a][m][h], 0, 0, 0);
      }
  };

  load(0);
  store(0);
  __syncthreads();
#pragma unroll 1
  for (int g0 = 0; g0 < NS; g0 += 2) {
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int g = g0 + e;
      if (g >= NS) break;
      load(g + 1);
#pragma unroll
      for (int c = 0; c < CB; c++)
        if (CB == 1 || g * CB + c < KB) step1(e, c);
      __builtin_amdgcn_sched_barrier(0);
      store(e ^ 1);
      __syncthreads();
    }
  }

  /* accumulator 4 b' + r of lane (n = lane % 16, g = lane / 16) is weight row
   * 4 g + r, hidden row n, chain 8 q + 2 b' + h (H = 1: 4 q + b'); chain l's
   * 256 sums go to part[l] at 4 lane + r */
  float *part = (float *)lds;
#pragma unroll
  for (int f = 0; f < MT * NT; f += PH) {
    if (f) __syncthreads();
#pragma unroll
    for (int g = 0; g < PH; g++)
#pragma unroll
      for (int h = 0; h < H; h++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const f32x16 &v = acc[(f + g) / NT][(f + g) % NT][h];
          const int l = H == 2 ? 8 * wid + 2 * c + h : 4 * wid + c;
          *(float4 *)&part[(g * 32 + l) * 256 + 4 * lane] = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
        }
    __syncthreads();
    const int o = tid & 255, g = PH == 1 ? 0 : wid >> 2;
    float p[32];
#pragma unroll
    for (int l = 0; l < 32; l++) p[l] = part[(g * 32 + l) * 256 + o];
#pragma unroll
    for (int sn = 16; sn >= 1; sn >>= 1)
#pragma unroll
      for (int l = 0; l < sn; l++) p[l] = p[l] + p[l + sn];
    const int n = n0 + (f + g) % NT * LR_TILE + ((o >> 2) & 15);
    const int r = v0 + (f + g) / NT * LR_TILE + 4 * (o >> 6) + (o & 3);
    if (n < n_rows && r < V) y[(size_t)n * V + r] = d3s_f32_to_bf16_rn(p[0]);
  }
}

template <int MT, int NT, int H, int CB, int MINW>
void launch_tiles(const LinearArgs &la, hipStream_t s) {
  const int rem = la.V % (LR_TILE * MT);
  const int vmain = rem <= LR_REM ? la.V - rem : la.V;
  const int64_t vgroups = (int64_t)((vmain + LR_XCDS * LR_TILE * MT - 1) / (LR_XCDS * LR_TILE * MT)) * LR_XCDS;
  /* rows per launch: at most 2^22 workgroups */
  const int64_t most = vgroups ? ((int64_t)1 << 22) / vgroups * LR_TILE * NT : la.n_rows;
  for (int64_t r0 = 0; r0 < la.n_rows; r0 += most) {
    const int n = (int)(la.n_rows - r0 < most ? la.n_rows - r0 : most);
    const int ntiles = (n + LR_TILE * NT - 1) / (LR_TILE * NT);
    const int64_t extra = ((int64_t)(la.V - vmain) * n + 16 / H - 1) / (16 / H);
    hipLaunchKernelGGL((k_linear_rows<MT, NT, H, CB, MINW>), dim3((unsigned)(vgroups * ntiles + extra)),
                       dim3(WAVE * 8 / H), 0, s, la.x + (size_t)r0 * la.K, la.w, la.K, la.V, n, ntiles, vmain,
                       la.y + (size_t)r0 * la.V);
  }
}

}  // namespace

/* 32 x 32 tiles on eight waves (half the operand conversions per MFMA of
 * 16 x 16 on four) when they fill the CUs, else 16 x 16: four times the
 * workgroups.  [64, 2048] x [4097, 2048]: 15.5 us against 16.4 us, 256 rows
 * 46.5 against 52.0 us, but 16 rows 14.5 against 7.7 us (128 workgroups). */
void launch_linear_rows(const LinearArgs &la, hipStream_t s) {
  if ((int64_t)((la.n_rows + 31) / 32) * (la.V / 32) >= 256)
    launch_tiles<2, 2, 1, 2, 2>(la, s);
  else
    launch_tiles<1, 1, 2, 2, 4>(la, s);
}

}  // namespace d3s
