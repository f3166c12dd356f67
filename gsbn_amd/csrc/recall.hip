/*
 * recall.hip -- frozen-weight batched recall.
 *
 * A trained population with one recurrent projection recalls B cues in
 * lock-step.  Weights Wij and biases bj are frozen (the reference's recall
 * mode, prn = 0: Proj.cpp:310-363 leaves bj alone and Proj.cpp:365-479 adds
 * the stored Wij to the support without recomputing it), so per cue b and
 * step t only the population dynamics run:
 *
 *   Pop(t)    support from E_{t-1}, dsup, WTA soft-max, spikes
 *             (Pop.cpp:229-323, as the solver's population kernel),
 *   E_t     = E_{t-1} (1 - kepsc) + sum of W over the rows active at t
 *             (jxx decay then row additions, Proj.cpp:310-363, 365-479),
 *
 * a row being active at t when its source unit spiked at t - di - 2.  Each
 * cue starts from the population's initial state (dsup = log(1/M),
 * Pop.cpp:59), an empty delay queue and E = 0, and draws with Philox key
 * seed + b, population 0.
 *
 * Both modes run in recall_wave_kernel, several steps per launch, where it
 * covers the population (see gsbn_recall_new).  Two support paths:
 *   exact  float weights, the additions in the reference's ascending row
 *          order: identical to a single-cue run of the solver (and the
 *          oracle) with the same weights;
 *   mfma   the support of all cues as one product S_{t-d-2} W of the 0/1
 *          spike matrix (B x Nsrc, bf16) and W (Nsrc x N, bf16) on the
 *          gfx950 matrix cores with float accumulation, fused with the
 *          decay: E = E (1 - kepsc) + S W.  Needs one delay for all rows.
 */
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/gsbn_amd.h"
#include "dbuf.h"
#include "detfast.h"
#include "detmath.h"
#include "gsbn_core.h"
#include "philox.h"
#include "wave.h"

#define RE_THREADS_MAX 1024
#define RE_RING 64 /* spike-history slots; latency di + 2 <= 33 */
#define RE_ROWS_MAX 2048 /* active rows compacted into LDS per (HCU, cue) and step */

/* GEMM tiling: 256 x 256 output tile per workgroup of 16 waves (64 x 64
 * each, 2 x 2 blocks of 32 x 32), K in steps of 64, LDS rows padded by 8 bf16 */
#define GM_BM 256
#define GM_BN 256
#define GM_BK 64
#define GM_GROUP 8
/* tiles of 64 x 64 below this many of 256 x 256, half the device's CUs (64 and
 * 256, us): 1 tile 4.6, 11; 12: 6.8, 28; 48 (1000 x 3000): 34, 76; 96 (8000 x
 * 700): 21, 31; 144 (3000 x 3000): 87, 78; 384 (8000 x 3000): 221, 160 */
#define GM_SMALL 128
/* the order in which the eight MFMAs of a 16-deep step issue with the LDS
 * reads of the next step, and with LDS writes and memory loads */
#define GM_MFMA __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#define GM_RD(n) __builtin_amdgcn_sched_group_barrier(0x100, n, 0);
#define GM_WR(n) __builtin_amdgcn_sched_group_barrier(0x200, n, 0);
#define GM_LD(n) __builtin_amdgcn_sched_group_barrier(0x020, n, 0);
#define GM_ORDER_READS \
  GM_MFMA GM_MFMA GM_RD(1) GM_MFMA GM_RD(1) GM_MFMA GM_RD(1) GM_MFMA GM_MFMA GM_RD(1) GM_MFMA GM_RD(1) \
  GM_MFMA GM_RD(1)
#define GM_ORDER_ALL                                                                              \
  GM_MFMA GM_RD(2) GM_MFMA GM_RD(3) GM_MFMA GM_RD(1) GM_WR(2) GM_MFMA GM_WR(3) GM_MFMA GM_WR(2)   \
  GM_MFMA GM_WR(1) GM_LD(2) GM_MFMA GM_LD(3) GM_MFMA GM_LD(3)

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 gsbn_bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float gsbn_f32x16;

namespace {

struct ReArgs {
  int B, Bp, H, M, C, N, Kp, W, dmin, dmax, count_from, mode;
  uint64_t seed;
  float taumdt, wtagain, maxfqdt, igain, wgain, lgbias, snoise, kepsc, lg_on, lg_off;
  float* dsup;            /* [B][N] */
  float* epsc;            /* [B][N] */
  int32_t* count;         /* [B][N] */
  const float* bj;        /* [N] */
  const float* wij;       /* [H*C*M] (exact) */
  const int32_t* di;      /* [H*C] */
  const int32_t* inv_off; /* [H][N+1] */
  const int32_t* inv_slot;
  int32_t* spk_cnt;       /* [RE_RING][B][H] */
  uint16_t* spk_list;     /* [RE_RING][B][H][M] */
  uint16_t* S;            /* [RE_RING][B][Kp] bf16 0/1 (mfma) */
  const int16_t* clamp;   /* [B][H] */
  const float* wmask;     /* [B][H] */
  int8_t* raster;         /* spikes, [steps kept][B][N] from step raster_t0, or NULL */
  /* the wave kernel (recall_wave_kernel) */
  int R, L, raster_t0, Np;
  float dsup0;
  const int32_t* one;     /* [H][N] slot of a source in an HCU: -1 none, -2 several (exact) */
  const uint16_t* Wb;     /* [H][N][M] bf16 weights by source (mfma) */
  const uint16_t* WT;     /* [Np][Kp] bf16 weights by destination unit (mfma) */
  int32_t* src_cnt;       /* [R][B] spikes of a step */
  uint16_t* src_list;     /* [R][B][N] their units, in no order */
  int32_t* out_idx;       /* [B][H] */
  int32_t* out_cnt;
};

inline int ret(hipError_t e) { return e == hipSuccess ? 0 : (int)e; }

/* exclusive prefix sum across the workgroup (blockDim a multiple of 64,
 * sh: blockDim / 64 ints), with the total */
__device__ __forceinline__ int block_scan_fast_re(int v, int* sh, int* total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int x = (int)wave_incl_scan((uint32_t)v);
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  int base = 0, tot = 0;
  for (int w = 0; w < nw; ++w) {
    const int t = sh[w];
    if (w < wid) base += t;
    tot += t;
  }
  *total = tot;
  __syncthreads();
  return base + x - v;
}

/* one workgroup per (HCU, cue): the population step and, in the exact mode,
 * the support update of that HCU's units */
__global__ void __launch_bounds__(RE_THREADS_MAX) recall_step_kernel(ReArgs a, int t) {
  extern __shared__ uint32_t sh_bits[];
  __shared__ __attribute__((aligned(16))) float sh_f[RE_THREADS_MAX];
  __shared__ int sh_scan[RE_THREADS_MAX / 64 + 1];
  __shared__ float sh_vsum;
  const int h = blockIdx.x, b = blockIdx.y, j = threadIdx.x;
  const int M = a.M, N = a.N;
  const bool live = j < M;
  const int n = h * M + j;
  const int64_t bn = (int64_t)b * N + n;

  /* support, dsup (Pop.cpp:229-261) */
  float u = 0.0f, dsup = 0.0f, E = 0.0f;
  if (live) {
    float z;
    gsbn_draw_unit_guarded(a.seed + (uint64_t)b, 0u, (uint32_t)t, (uint32_t)n, &u, &z);
    const float xi = a.snoise * z;
    E = a.epsc[bn];
    float wsup = 0.0f;
    wsup += a.bj[n] + E;
    const float lginp = (a.clamp[(int64_t)b * a.H + h] == j) ? a.lg_on : a.lg_off;
    float sup = a.lgbias + a.igain * lginp + xi;
    sup += (a.wgain * a.wmask[(int64_t)b * a.H + h]) * wsup;
    const float d0 = a.dsup[bn];
    dsup = d0 + (sup - d0) * a.taumdt;
    a.dsup[bn] = dsup;
  }
  /* WTA maximum: first of equal maxima, as the sequential reference */
  {
    const float mv = wave_max_left(live ? dsup : -INFINITY);
    if ((j & 63) == 0) sh_f[j >> 6] = mv;
  }
  __syncthreads();
  float maxdsup = sh_f[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
    const float o = sh_f[w];
    if (o > maxdsup) maxdsup = o;
  }
  __syncthreads();
  /* soft-max (Pop.cpp:280-302) */
  const float maxact = gsbn_expf_guarded(a.wtagain * maxdsup);
  float act = 0.0f;
  if (live) {
    act = gsbn_expf_guarded(a.wtagain * (dsup - maxdsup));
    if (maxact < 1.0f) act *= maxact;
    sh_f[j] = act;
  }
  __syncthreads();
  if (j == 0) sh_vsum = ordered_sum_lds(sh_f, M);
  __syncthreads();
  if (live && sh_vsum > 1.0f) act /= sh_vsum;
  /* spikes (Pop.cpp:305-323) */
  const int spk = (live && u < act * a.maxfqdt) ? 1 : 0;
  if (live) {
    if (t > a.count_from) a.count[bn] += spk;
    if (a.raster) a.raster[bn] = (int8_t)spk;
  }
  const int slot = t % RE_RING;
  if (a.mode == GSBN_RECALL_MFMA) {
    if (live) a.S[((int64_t)slot * a.Bp + b) * a.Kp + n] = spk ? (uint16_t)0x3F80u : (uint16_t)0u;
    return;
  }
  /* spike list of this HCU (ascending) for the queue of later steps */
  {
    const int lane = j & 63, wid = j >> 6, nw = blockDim.x >> 6;
    const uint64_t bal = __ballot(spk);
    const int before = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0) sh_scan[wid] = __popcll(bal);
    __syncthreads();
    int base = 0, tot = 0;
    for (int w = 0; w < nw; ++w) {
      if (w < wid) base += sh_scan[w];
      tot += sh_scan[w];
    }
    const int64_t lb = ((int64_t)slot * a.B + b) * a.H + h;
    if (spk) a.spk_list[lb * M + base + before] = (uint16_t)j;
    if (j == 0) a.spk_cnt[lb] = tot;
  }
  /* exact support update: E (1 - kepsc), then + Wij of every row active at
   * t in ascending row order (Proj.cpp:310-363 then 365-479) */
  const int C = a.C, Wd = a.W;
  for (int w = j; w < Wd; w += blockDim.x) sh_bits[w] = 0u;
  __syncthreads();
  const int32_t* off = a.inv_off + (int64_t)h * (N + 1);
  for (int d = a.dmin; d <= a.dmax; ++d) {
    const int s = t - d - 2;
    if (s < 1) continue;
    const int ss = s % RE_RING;
    const int32_t* cnts = a.spk_cnt + ((int64_t)ss * a.B + b) * a.H;
    const uint16_t* lsts = a.spk_list + ((int64_t)ss * a.B + b) * a.H * M;
    for (int hs = j; hs < a.H; hs += blockDim.x) {
      const int c = cnts[hs];
      for (int i = 0; i < c; ++i) {
        const int src = hs * M + lsts[(int64_t)hs * M + i];
        for (int q = off[src]; q < off[src + 1]; ++q) {
          const int k = a.inv_slot[q];
          if (a.di[(int64_t)h * C + k] == d) atomicOr(&sh_bits[k >> 5], 1u << (k & 31));
        }
      }
    }
  }
  __syncthreads();
  /* the active rows in ascending order, compacted into LDS (after the bitmap
   * in the dynamic LDS), so each thread can have eight weight loads in
   * flight instead of one per row; more than RE_ROWS_MAX rows (not reached
   * by recall, whose active rows are the few spiking sources) fall back to
   * walking the bitmap */
  int* const sh_rows = reinterpret_cast<int*>(sh_bits + Wd);
  int nrows;
  {
    const int per = (Wd + (int)blockDim.x - 1) / (int)blockDim.x;
    const int w0 = j * per;
    const int w1 = w0 + per < Wd ? w0 + per : Wd;
    int c = 0;
    for (int w = w0; w < w1; ++w) c += __popc(sh_bits[w]);
    int pos = block_scan_fast_re(c, sh_scan, &nrows);
    if (nrows <= RE_ROWS_MAX) {
      for (int w = w0; w < w1; ++w) {
        uint32_t bits = sh_bits[w];
        while (bits) {
          sh_rows[pos++] = (w << 5) + __ffs(bits) - 1;
          bits &= bits - 1;
        }
      }
    }
    __syncthreads();
  }
  if (live) {
    float e = E * (1 - a.kepsc);
    const float* wrow = a.wij + (int64_t)h * C * M + j;
    if (nrows <= RE_ROWS_MAX) {
      for (int r = 0; r < nrows; r += 8) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = r + q < nrows ? wrow[(int64_t)sh_rows[r + q] * M] : 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (r + q < nrows) e = e + v[q];
      }
    } else {
      for (int w = 0; w < Wd; ++w) {
        uint32_t bits = sh_bits[w];
        while (bits) {
          const int k = (w << 5) + __ffs(bits) - 1;
          bits &= bits - 1;
          e = e + wrow[(int64_t)k * M];
        }
      }
    }
    a.epsc[bn] = e;
  }
}

/* The population step of the mfma mode with one wave per (HCU, cue) and
 * four pairs per workgroup: lane l takes units l, l + 64, ... (UPL per
 * lane), so no workgroup barrier is needed and a hypercolumn of M <= 64 * UPL
 * units occupies one wave instead of ceil(M / 64).  Same operations per unit
 * as recall_step_kernel: the WTA maximum combines the 64-unit ranges left to
 * right with the sequential comparison, and the normaliser is summed in
 * ascending unit order by lane 0 from the wave's LDS row. */
template <int UPL>
__global__ void __launch_bounds__(256) recall_pop_wave_kernel(ReArgs a, int t) {
  __shared__ __attribute__((aligned(16))) float sh_act[4][UPL * 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t pair = (int64_t)blockIdx.x * 4 + wave; /* b * H + h */
  if (pair >= (int64_t)a.B * a.H) return;              /* uniform per wave */
  const int b = (int)(pair / a.H), h = (int)(pair - (int64_t)b * a.H);
  const int M = a.M, N = a.N;
  const int cl = a.clamp[pair];
  const float wm = a.wmask[pair];
  float* const row = sh_act[wave];
  float dsup[UPL], u[UPL];
  int cnt[UPL];
  /* support, dsup (Pop.cpp:229-261) */
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    const int j = lane + 64 * i;
    dsup[i] = 0.0f;
    u[i] = 0.0f;
    cnt[i] = 0;
    if (j < M) {
      const int n = h * M + j;
      const int64_t bn = (int64_t)b * N + n;
      const float E = a.epsc[bn];
      const float bjv = a.bj[n];
      const float d0 = a.dsup[bn];
      if (t > a.count_from) cnt[i] = a.count[bn];
      float z;
      gsbn_draw_unit_guarded(a.seed + (uint64_t)b, 0u, (uint32_t)t, (uint32_t)n, &u[i], &z);
      const float xi = a.snoise * z;
      float wsup = 0.0f;
      wsup += bjv + E;
      const float lginp = cl == j ? a.lg_on : a.lg_off;
      float sup = a.lgbias + a.igain * lginp + xi;
      sup += (a.wgain * wm) * wsup;
      dsup[i] = d0 + (sup - d0) * a.taumdt;
      a.dsup[bn] = dsup[i];
    }
  }
  /* WTA maximum: each 64-unit range by shuffles, the ranges left to right */
  float maxdsup = 0.0f;
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    const float mv = wave_max_left(lane + 64 * i < M ? dsup[i] : -INFINITY);
    if (i == 0) {
      maxdsup = mv;
    } else if (64 * i < M && mv > maxdsup) {
      maxdsup = mv;
    }
  }
  /* soft-max (Pop.cpp:280-302) */
  const float maxact = gsbn_expf_guarded(a.wtagain * maxdsup);
  float act[UPL];
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    act[i] = 0.0f;
    if (lane + 64 * i < M) {
      act[i] = gsbn_expf_guarded(a.wtagain * (dsup[i] - maxdsup));
      if (maxact < 1.0f) act[i] *= maxact;
      row[lane + 64 * i] = act[i];
    }
  }
  float vsum = 0.0f;
  if (lane == 0) vsum = ordered_sum_lds(row, M);
  vsum = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(vsum)));
  /* spikes (Pop.cpp:305-323) */
  const int slot = t % RE_RING;
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    const int j = lane + 64 * i;
    if (j >= M) continue;
    float ac = act[i];
    if (vsum > 1.0f) ac /= vsum;
    const int spk = u[i] < ac * a.maxfqdt ? 1 : 0;
    const int n = h * M + j;
    const int64_t bn = (int64_t)b * N + n;
    if (t > a.count_from) a.count[bn] = cnt[i] + spk;
    if (a.raster) a.raster[bn] = (int8_t)spk;
    a.S[((int64_t)slot * a.Bp + b) * a.Kp + n] = spk ? (uint16_t)0x3F80u : (uint16_t)0u;
  }
}

#define RW_WAVES 4 /* cues per workgroup of recall_wave_kernel */

/* acc[u] (unit lane + 64 u) += W's 16-source block `blk`, sources of `bits`,
 * by the matrix instruction of spike_gemm_kernel on the same operands: rows 0
 * and 4 of the A block hold the cue, so accumulator 0 of a lane (row 0 for
 * lanes 0-31, row 4 for lanes 32-63) is that lane's unit of the column block.
 * Called by whole waves. */
template <int UPL>
__device__ __forceinline__ void add_block_mfma(const ReArgs& a, int h, int blk, uint32_t bits,
                                               int lane, float* acc) {
  union {
    gsbn_bf16x8 v;
    uint16_t u[8];
  } A;
  const uint32_t mine = (lane & 27) == 0 ? (bits >> ((lane >> 5) * 8)) & 0xffu : 0u;
#pragma unroll
  for (int q = 0; q < 8; ++q) A.u[q] = ((mine >> q) & 1u) ? (uint16_t)0x3F80u : (uint16_t)0u;
#pragma unroll
  for (int u = 0; u < UPL; ++u) {
    float r[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      int n = h * a.M + 64 * u + 32 * c + (lane & 31);
      n = n < a.Np ? n : a.Np - 1;
      const gsbn_bf16x8 B = *reinterpret_cast<const gsbn_bf16x8*>(
          a.WT + (int64_t)n * a.Kp + blk * 16 + (lane >> 5) * 8);
      gsbn_f32x16 C;
#pragma unroll
      for (int q = 0; q < 16; ++q) C[q] = 0.0f;
      C[0] = acc[u];
      C = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A.v, B, C, 0, 0, 0);
      r[c] = C[0];
      /* one block's accumulators at a time */
      __builtin_amdgcn_sched_barrier(0);
    }
    acc[u] = lane < 32 ? r[0] : r[1];
  }
}

/* Steps t0 .. t0 + nt - 1 of the recall, one wave per (HCU, cue), UPL units
 * per lane.  A row active at t has a source that spiked at t - di - 2, so
 * the steps of a run of L = dmin + 2 read only spikes of earlier launches:
 * a wave keeps its pair's state in registers for L steps.  Per step: the
 * population update (Pop.cpp:229-323), the spikes appended to the cue's list
 * of the step, and the support update from the cue's list of step t - d - 2:
 * its sources' rows sorted by rank (at most 64; more, or several delays or
 * slots per source, go through bitmap windows), weights read row by row.
 *   exact: E = E (1 - kepsc), then + Wij of each row in ascending row order.
 *   mfma (BF): E = E (1 - kepsc) + SW, SW with the bits of the dense product:
 *   that product adds, 16 sources at a time, mostly zeros, which change
 *   nothing; where every sum of the nonzero terms is exact (one term per
 *   block, s - a == b and s - b == a) its value is the float sum, and
 *   otherwise the nonzero blocks go through the same matrix instruction.
 *
 * What bounds it: issue (Philox and the double sequences of the draw and the
 * soft-max): 630 vector instructions per step of up to 128 units, the vector
 * units 85 % busy (mfma 670, 72 %).  Hence one wave per
 * pair without idle waves, the normalisers of a workgroup's pairs summed by
 * as many lanes at once (100 dependent additions for one lane would
 * be 400 issue cycles per pair), and the maximum's exponential evaluated by
 * the lane that holds the maximum, whose own is 1.  Workgroup i runs on XCD
 * i % 8: an XCD takes one HCU at a time for all cues, so that the HCU's
 * weights (4 MB at 100 x 100) stay in its L2.  Four waves per workgroup and
 * six waves per SIMD for exact (eight and four: 68.5 ms); the mfma form's
 * accumulators hold it at four.
 * 8192 cues x 50 steps at 100 x 100: exact 54.5 ms (a workgroup per pair and
 * one step per launch: 107 ms with the same short sequences), mfma 68.5 ms
 * (dense product 75 ms and population step 43 ms: 120 ms); one cue at 10 x 10:
 * 0.24 ms (0.94 ms). */
template <int UPL, bool BF>
__global__ void __launch_bounds__(64 * RW_WAVES, BF ? (UPL == 1 ? 5 : UPL == 2 ? 4 : 3) : UPL <= 2 ? 6 : 4)
    recall_wave_kernel(ReArgs a, int t0, int nt, int last) {
  __shared__ __attribute__((aligned(16))) float sh_act[RW_WAVES][64 * UPL + 4];
  __shared__ float sh_sum[RW_WAVES];
  __shared__ uint32_t sh_bm[RW_WAVES][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nb8 = (a.B + RW_WAVES - 1) / RW_WAVES;
  const int xcd = blockIdx.x & 7, bi = blockIdx.x >> 3;
  const int h = xcd + 8 * (bi / nb8);
  if (h >= a.H) return; /* the whole workgroup */
  const int b = (bi % nb8) * RW_WAVES + wave;
  const bool on = b < a.B; /* uniform per wave; the others only meet the barriers */
  const int M = a.M, N = a.N, B = a.B;
  const int64_t pair = (int64_t)b * a.H + h;
  const int64_t bn0 = (int64_t)b * N + (int64_t)h * M;

  float dsup[UPL], E[UPL], bjv[UPL];
  int cnt[UPL];
  int cl = -1;
  float wm = 0.0f;
  if (on) {
    cl = a.clamp[pair];
    wm = a.wmask[pair];
#pragma unroll
    for (int i = 0; i < UPL; ++i) {
      const int j = lane + 64 * i;
      dsup[i] = a.dsup0;
      E[i] = 0.0f;
      cnt[i] = 0;
      bjv[i] = 0.0f;
      if (j < M) {
        bjv[i] = a.bj[h * M + j];
        if (t0 > 1) {
          dsup[i] = a.dsup[bn0 + j];
          E[i] = a.epsc[bn0 + j];
          cnt[i] = a.count[bn0 + j];
        }
      }
    }
    /* the counters of the next launch's steps (their slots' previous steps
     * are no longer read) */
    if (h == 0 && lane < a.L) a.src_cnt[(int64_t)((t0 + nt + lane) % a.R) * B + b] = 0;
  }
  const bool single = a.dmin == a.dmax;

  for (int t = t0; t < t0 + nt; ++t) {
    /* the sources active at t and their rows, looked up before the draws */
    int nsrc = 0, key = -1;
    bool general = false;
    if (on && single) {
      const int s = t - a.dmin - 2;
      if (s >= 1) {
        const int64_t sb = (int64_t)(s % a.R) * B + b;
        nsrc = __builtin_amdgcn_readfirstlane(a.src_cnt[sb]);
        general = nsrc > 64;
        if (!general && lane < nsrc) {
          const int src = a.src_list[sb * N + lane];
          key = BF ? src : a.one[(int64_t)h * N + src];
        }
      }
    } else if (on) {
      general = a.dmax > 0;
    }
    float u[UPL], act[UPL];
    if (on) {
      /* support, dsup (Pop.cpp:229-261) */
#pragma unroll
      for (int i = 0; i < UPL; ++i) {
        const int j = lane + 64 * i;
        float z;
        gsbn_draw_unit_guarded(a.seed + (uint64_t)b, 0u, (uint32_t)t, (uint32_t)(h * M + j), &u[i], &z);
        const float xi = a.snoise * z;
        float wsup = 0.0f;
        wsup += bjv[i] + E[i];
        const float lginp = cl == j ? a.lg_on : a.lg_off;
        float sup = a.lgbias + a.igain * lginp + xi;
        sup += (a.wgain * wm) * wsup;
        dsup[i] = dsup[i] + (sup - dsup[i]) * a.taumdt;
      }
      /* WTA maximum: each 64-unit range by a wave scan, left to right */
      float maxdsup = 0.0f;
#pragma unroll
      for (int i = 0; i < UPL; ++i) {
        const float mv = wave_max_left(lane + 64 * i < M ? dsup[i] : -INFINITY);
        if (i == 0) {
          maxdsup = mv;
        } else if (64 * i < M && mv > maxdsup) {
          maxdsup = mv;
        }
      }
      /* soft-max (Pop.cpp:280-302).  exp(wtagain * maxdsup) comes from a lane
       * whose dsup is the maximum (its own activity is exp(0) = 1); without
       * one (NaN), or with an infinite gain, it is evaluated by itself */
      const float xmax = a.wtagain * maxdsup;
      float maxact = 0.0f;
      bool have = false;
#pragma unroll
      for (int i = 0; i < UPL; ++i) {
        const float diff = dsup[i] - maxdsup;
        const bool top = lane + 64 * i < M && diff == 0.0f && a.wtagain * diff == 0.0f;
        const float e = gsbn_expf_guarded(top ? xmax : a.wtagain * diff);
        act[i] = top ? 1.0f : e;
        const uint64_t tb = __ballot(top);
        if (tb && !have) {
          maxact = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), __builtin_ctzll(tb)));
          have = true;
        }
      }
      if (!have) maxact = gsbn_expf_guarded(xmax);
#pragma unroll
      for (int i = 0; i < UPL; ++i) {
        if (maxact < 1.0f) act[i] *= maxact;
        sh_act[wave][lane + 64 * i] = act[i];
      }
    }
    __syncthreads();
    if (threadIdx.x < RW_WAVES) sh_sum[threadIdx.x] = ordered_sum_lds(sh_act[threadIdx.x], M);
    __syncthreads();
    if (!on) continue;
    const float vsum = sh_sum[wave];
    /* spikes (Pop.cpp:305-323), appended to the cue's list of this step */
    int spk[UPL], tot = 0, before[UPL];
#pragma unroll
    for (int i = 0; i < UPL; ++i) {
      const int j = lane + 64 * i;
      float ac = act[i];
      if (vsum > 1.0f) ac /= vsum;
      spk[i] = (j < M && u[i] < ac * a.maxfqdt) ? 1 : 0;
      const uint64_t bal = __ballot(spk[i]);
      before[i] = tot + __popcll(bal & ((1ull << lane) - 1ull));
      tot += __popcll(bal);
      if (t > a.count_from) cnt[i] += spk[i];
      if (a.raster && j < M) a.raster[(int64_t)(t - a.raster_t0) * B * N + bn0 + j] = (int8_t)spk[i];
    }
    if (tot) {
      const int64_t sb = (int64_t)(t % a.R) * B + b;
      int base = 0;
      if (lane == 0) base = atomicAdd(&a.src_cnt[sb], tot);
      base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
      for (int i = 0; i < UPL; ++i)
        if (spk[i]) a.src_list[sb * N + base + before[i]] = (uint16_t)(h * M + lane + 64 * i);
    }
    /* support update */
    float e[UPL];
#pragma unroll
    for (int i = 0; i < UPL; ++i) e[i] = BF ? 0.0f : E[i] * (1 - a.kepsc);
    if (!BF && __ballot(key == -2)) general = true;
    if (!general) {
      const uint64_t m = __ballot(key >= 0);
      const int nk = __popcll(m);
      if (nk) {
        /* ascending keys: lane r holds the r-th */
        int rank = 0;
        for (uint64_t mm = m; mm; mm &= mm - 1)
          rank += __builtin_amdgcn_readlane(key, __builtin_ctzll(mm)) < key;
        if (key < 0) rank = nk + __popcll(~m & ((1ull << lane) - 1ull));
        const int ks = __builtin_amdgcn_ds_permute(rank << 2, key);
        bool exactly = true;
        if (BF) {
          const int nx = __builtin_amdgcn_ds_bpermute(((lane + 1) & 63) << 2, ks);
          if (__ballot(lane + 1 < nk && (nx >> 4) == (ks >> 4))) exactly = false;
        }
        if (exactly) {
          bool off = false;
          const int64_t hrow = (int64_t)h * (BF ? N : a.C);
          constexpr int G = UPL <= 2 ? 8 : 4;
          for (int r = 0; r < nk; r += G) {
            float v[G][UPL];
#pragma unroll
            for (int q = 0; q < G; ++q) {
              const int k = __builtin_amdgcn_readlane(ks, r + q < nk ? r + q : nk - 1);
              const int64_t at = (hrow + k) * M;
#pragma unroll
              for (int i = 0; i < UPL; ++i) {
                int j = lane + 64 * i;
                j = j < M ? j : M - 1;
                v[q][i] = BF ? __uint_as_float((uint32_t)a.Wb[at + j] << 16) : a.wij[at + j];
              }
            }
#pragma unroll
            for (int q = 0; q < G; ++q) {
              if (r + q < nk) {
#pragma unroll
                for (int i = 0; i < UPL; ++i) {
                  const float s = e[i] + v[q][i];
                  if (BF) off = off || !(s - e[i] == v[q][i] && s - v[q][i] == e[i]);
                  e[i] = s;
                }
              }
            }
          }
          if (BF && __ballot(off)) exactly = false;
        }
        if (BF && !exactly) {
#pragma unroll
          for (int i = 0; i < UPL; ++i) e[i] = 0.0f;
          for (int r = 0; r < nk;) {
            const int blk = __builtin_amdgcn_readlane(ks, r) >> 4;
            uint32_t bits = 0;
            int k;
            while (r < nk && ((k = __builtin_amdgcn_readlane(ks, r)) >> 4) == blk) {
              bits |= 1u << (k & 15);
              ++r;
            }
            add_block_mfma<UPL>(a, h, blk, bits, lane, e);
          }
        }
      }
    } else {
      /* any number of rows: windows of 2048 keys (slots, or sources) */
      const int span = BF ? N : a.C;
      for (int w0 = 0; w0 < span; w0 += 2048) {
        sh_bm[wave][lane] = 0u;
        wave_order();
        for (int d = a.dmin; d <= a.dmax; ++d) {
          const int s = t - d - 2;
          if (s < 1) break;
          const int64_t sb = (int64_t)(s % a.R) * B + b;
          const int n = __builtin_amdgcn_readfirstlane(a.src_cnt[sb]);
          for (int i = lane; i < n; i += 64) {
            const int src = a.src_list[sb * N + i];
            if (BF) {
              const int k = src - w0;
              if (k >= 0 && k < 2048) atomicOr(&sh_bm[wave][k >> 5], 1u << (k & 31));
            } else {
              const int32_t* off = a.inv_off + (int64_t)h * (N + 1);
              for (int q = off[src]; q < off[src + 1]; ++q) {
                const int slot = a.inv_slot[q], k = slot - w0;
                if (k >= 0 && k < 2048 && a.di[(int64_t)h * a.C + slot] == d)
                  atomicOr(&sh_bm[wave][k >> 5], 1u << (k & 31));
              }
            }
          }
        }
        wave_order();
        const int word = (int)sh_bm[wave][lane];
        wave_order();
        for (uint64_t nz = __ballot(word != 0); nz; nz &= nz - 1) {
          const int l = __builtin_ctzll(nz);
          uint32_t bits = (uint32_t)__builtin_amdgcn_readlane(word, l);
          const int k0 = w0 + 32 * l;
          if (BF) {
            if (bits & 0xffffu) add_block_mfma<UPL>(a, h, k0 >> 4, bits & 0xffffu, lane, e);
            if (bits >> 16) add_block_mfma<UPL>(a, h, (k0 >> 4) + 1, bits >> 16, lane, e);
          } else {
            while (bits) {
              const int64_t at = ((int64_t)h * a.C + k0 + __builtin_ctz(bits)) * M;
              bits &= bits - 1;
#pragma unroll
              for (int i = 0; i < UPL; ++i) {
                const int j = lane + 64 * i;
                e[i] = e[i] + a.wij[at + (j < M ? j : M - 1)];
              }
            }
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < UPL; ++i) E[i] = BF ? (1 - a.kepsc) * E[i] + e[i] : e[i];
  }
  if (!on) return;
  if (!last) {
#pragma unroll
    for (int i = 0; i < UPL; ++i) {
      const int j = lane + 64 * i;
      if (j < M) {
        a.dsup[bn0 + j] = dsup[i];
        a.epsc[bn0 + j] = E[i];
        a.count[bn0 + j] = cnt[i];
      }
    }
    return;
  }
  /* first strict maximum of the counts (ProcCheck/Pop.cpp:35-50) */
  int mc = 0;
#pragma unroll
  for (int i = 0; i < UPL; ++i) mc = max(mc, lane + 64 * i < M ? cnt[i] : 0);
  for (int o = 32; o; o >>= 1) mc = max(mc, __shfl_xor(mc, o));
  int mi = -1;
#pragma unroll
  for (int i = 0; i < UPL; ++i) {
    const uint64_t bal = __ballot(lane + 64 * i < M && cnt[i] == mc);
    if (mi < 0 && mc > 0 && bal) mi = 64 * i + __builtin_ctzll(bal);
  }
  if (lane == 0) {
    a.out_idx[pair] = mi;
    a.out_cnt[pair] = mc;
  }
}

/* the slot of every (HCU, source): -1 without one, -2 with several.  (Made on
 * the host and uploaded, this was 0.5 of the 17 ms that a handle of 100 x 100
 * took to build.) */
__global__ void recall_one_kernel(int64_t n, int N, const int32_t* inv_off, const int32_t* inv_slot,
                                  int32_t* one) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t h = i / N;
    const int32_t* o = inv_off + h * (N + 1) + (i - h * N);
    const int q0 = o[0], q1 = o[1];
    one[i] = q1 == q0 ? -1 : q1 == q0 + 1 ? inv_slot[q0] : -2;
  }
}

/* bf16 weights of the mfma mode from the float weights: one workgroup per
 * (HCU, source), the source's slots summed in double in ascending order
 * (CSR), stored by source (Wb, where given) and by destination unit (WT);
 * *nonfinite is set when one is infinite or NaN. */
__global__ void recall_weights_kernel(int H, int M, int C, int N, int Kp, const float* wij,
                                      const int32_t* inv_off, const int32_t* inv_slot, uint16_t* Wb,
                                      uint16_t* WT, int32_t* nonfinite) {
  const int src = blockIdx.x;
  for (int h = blockIdx.y; h < H; h += gridDim.y) {
    const int32_t* off = inv_off + (int64_t)h * (N + 1);
    const int q0 = off[src], q1 = off[src + 1];
    for (int j = threadIdx.x; j < M; j += blockDim.x) {
      double acc = 0.0;
      for (int q = q0; q < q1; ++q)
        acc += (double)wij[((int64_t)h * C + inv_slot[q]) * M + j];
      const uint16_t v = gsbn_f32_to_bf16((float)acc);
      if ((v & 0x7f80u) == 0x7f80u) *nonfinite = 1;
      if (Wb) Wb[((int64_t)h * N + src) * M + j] = v;
      WT[((int64_t)h * M + j) * Kp + src] = v;
    }
  }
}

/* E[b][n] = beta E[b][n] + sum_k S[b][k] WT[n][k]: bf16 inputs, float
 * accumulation on v_mfma_f32_32x32x16_bf16, k ascending.  S and WT have Kp
 * columns (Kp a multiple of GM_BK, zero padded); S has ceil(B / GM_BM) * GM_BM
 * rows and WT ceil(N / GM_BN) * GM_BN rows, so tiles never read past them.
 *
 * Large products (few tiles take 64 x 64, four waves of 32 x 32): a 256 x 256
 * output tile per workgroup of 8 waves (128 x 64 each: 4 x 2 MFMA blocks, 6
 * LDS reads of 16 bytes per 8 MFMAs, where 64 x 64 takes 8), K in steps of 64
 * through two LDS buffers.  While the products of one K tile run, the next
 * goes from registers to the other buffer and the one after that is loaded: a
 * full K tile (1.6 us) for the loads to arrive, one barrier per K tile, behind
 * which the last quarter of its products issues together with the first reads
 * of the next.  Chunks are permuted within a row instead of padding (no bank
 * conflicts; with r % 8 for r / 2 % 8, 3 of 8 LDS cycles were conflicts), and
 * the MFMAs are interleaved with the rest (without: 1.44 ms).  Workgroup i
 * runs on XCD i % 8: each XCD has consecutive tiles, in groups of GM_GROUP row
 * tiles, so that its 32 workgroups share 8 + 4 tiles of operands per K step
 * instead of 32 + 1.
 * What bounds it: the clock under this load (2.0-2.2 GHz), with the matrix
 * units 59 % busy; the rest is barrier skew and the tile's end, with one
 * workgroup per CU.  8192 x 10000 x 10048: 1.27-1.28 ms, 1.28 PFLOP/s (1.60 ms
 * with 16 waves of 64 x 64, one buffer and E read and written value by value;
 * a vendor library's product takes 1.26 ms).  16 waves of 64 x 64 in this form
 * 1.28 ms, K steps of 32 1.39, 128 x 256 tiles and two workgroups per CU 1.65,
 * 128 x 128 2.6, 4 waves of 128 x 128 1.54. */
template <int BM, int BN, int WM, int WN> /* tile, waves down and across it */
__global__ void __launch_bounds__(64 * WM * WN)
    spike_gemm_kernel(const uint16_t* __restrict__ S, const uint16_t* __restrict__ WT,
                      float* __restrict__ E, int Bn, int N, int Kp, float beta, int mtiles,
                      int ntiles) {
  constexpr int TM = BM / WM, TN = BN / WN, MI = TM / 32, NI = TN / 32;
  constexpr int RP = 8 * WM * WN, NC = BM / RP; /* staged rows per pass, passes */
  constexpr bool ORDER = MI == 4 && NI == 2 && NC == 4;
  static_assert(BM == BN && GM_BK == 64 && RP % 16 == 0, "staging");
  __shared__ __attribute__((aligned(16))) uint16_t sa[2][BM * GM_BK], sb[2][BN * GM_BK];
  const int nwg = mtiles * ntiles;
  /* tiles of one XCD (workgroup i runs on XCD i % 8) are consecutive; there
   * they go down GM_GROUP row tiles before the next column tile */
  int mt, nt;
  {
    const int x = blockIdx.x & 7, q = nwg >> 3, r = nwg & 7;
    const int i = x * q + (x < r ? x : r) + (blockIdx.x >> 3);
    const int grp = i / (GM_GROUP * ntiles), in = i - grp * GM_GROUP * ntiles;
    const int rows = mtiles - grp * GM_GROUP < GM_GROUP ? mtiles - grp * GM_GROUP : GM_GROUP;
    nt = in / rows;
    mt = grp * GM_GROUP + in - nt * rows;
  }
  const int m0 = mt * BM, n0 = nt * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave - wm * WN;

  gsbn_f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int jj = 0; jj < NI; ++jj)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][jj][r] = 0.0f;

  /* 16-byte chunk c of row r of a tile lies at chunk c ^ (r / 2 % 8) of the
   * row: the 16 rows that a 256-byte LDS access reads lie in 64 banks */
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4))); /* uint4 would go to scratch */
  const int crow = tid >> 3, cc = tid & 7;
  const uint32_t voff = (uint32_t)crow * (uint32_t)Kp * 2u + (uint32_t)cc * 16u;
  const uint16_t* const pa = S + (int64_t)m0 * Kp;
  const uint16_t* const pb = WT + (int64_t)n0 * Kp;
  const int64_t rs = (int64_t)RP * Kp;
  const int wr = crow * GM_BK + ((cc ^ ((crow >> 1) & 7)) * 8);
  u32x4 ra[NC], rb[NC];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      ra[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(pa + i * rs + k0) + voff);
      rb[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(pb + i * rs + k0) + voff);
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      *reinterpret_cast<u32x4*>(&sa[buf][wr + i * RP * GM_BK]) = ra[i];
      *reinterpret_cast<u32x4*>(&sb[buf][wr + i * RP * GM_BK]) = rb[i];
    }
  };
  const int arow = (wm * TM + (lane & 31)) * GM_BK, brow = (wn * TN + (lane & 31)) * GM_BK;
  gsbn_bf16x8 af[2][MI], bf[2][NI];
  auto frags = [&](int buf, int ks, int set) {
    const int c = ((ks * 2 + (lane >> 5)) ^ ((lane >> 1) & 7)) * 8;
#pragma unroll
    for (int i = 0; i < MI; ++i)
      af[set][i] = *reinterpret_cast<const gsbn_bf16x8*>(&sa[buf][arow + i * 32 * GM_BK + c]);
#pragma unroll
    for (int jj = 0; jj < NI; ++jj)
      bf[set][jj] = *reinterpret_cast<const gsbn_bf16x8*>(&sb[buf][brow + jj * 32 * GM_BK + c]);
  };
  auto product = [&](int set) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int jj = 0; jj < NI; ++jj)
        acc[i][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[set][i], bf[set][jj], acc[i][jj], 0, 0, 0);
  };

  const int nk = Kp / GM_BK;
  fetch(0);
  put(0);
  fetch(nk > 1 ? GM_BK : 0);
  __syncthreads();
  frags(0, 0, 0);
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    frags(buf, 1, 1);
    product(0);
    if constexpr (ORDER) {
      GM_ORDER_READS
    }
    frags(buf, 2, 0);
    put(buf ^ 1);
    fetch((kt + 2 < nk ? kt + 2 : nk - 1) * GM_BK); /* past the last K tile: unused */
    product(1);
    if constexpr (ORDER) {
      GM_ORDER_ALL
    }
    frags(buf, 3, 1);
    product(0);
    if constexpr (ORDER) {
      GM_ORDER_READS
    }
    __syncthreads(); /* every wave has read this K tile and stored its part of the next */
    frags(buf ^ 1, 0, 0);
    product(1);
    if constexpr (ORDER) {
      GM_ORDER_READS
    }
  }
  /* accumulator r of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4 and
   * column l % 32 of its 32 x 32 block; a block's 16 values of E are read
   * before the first is written (one after the other, each waits for memory) */
  const bool inside = m0 + BM <= Bn && n0 + BN <= N; /* the whole tile */
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int jj = 0; jj < NI; ++jj) {
      const int col = n0 + wn * TN + jj * 32 + (lane & 31);
      const int row0 = m0 + wm * TM + i * 32 + (lane >> 5) * 4;
      float v[16];
      if (inside) {
        float* const p = E + (int64_t)row0 * N + col;
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = p[(int64_t)((r >> 2) * 8 + (r & 3)) * N];
#pragma unroll
        for (int r = 0; r < 16; ++r)
          p[(int64_t)((r >> 2) * 8 + (r & 3)) * N] = beta * v[r] + acc[i][jj][r];
      } else if (col < N) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = row0 + (r >> 2) * 8 + (r & 3);
          v[r] = E[(int64_t)(row < Bn ? row : Bn - 1) * N + col];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = row0 + (r >> 2) * 8 + (r & 3);
          if (row < Bn) E[(int64_t)row * N + col] = beta * v[r] + acc[i][jj][r];
        }
      }
    }
}

/* first strict maximum of each (cue, HCU)'s counts (ProcCheck/Pop.cpp:35-50) */
__global__ void recall_argmax_kernel(int B, int H, int M, const int32_t* count, int32_t* idx,
                                     int32_t* cnt) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (g >= (int64_t)B * H) return;
  int mi = -1, mc = 0;
  const int32_t* c = count + g * M;
  for (int j = 0; j < M; ++j) {
    if (c[j] > mc) {
      mi = j;
      mc = c[j];
    }
  }
  idx[g] = mi;
  cnt[g] = mc;
}

__global__ void re_fill_f32(float* p, int64_t n, float v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

int grid_of(int64_t n) {
  int64_t g = (n + 255) / 256;
  return (int)std::min<int64_t>(std::max<int64_t>(g, 1), 16384);
}

}  // namespace

namespace gsbn {
void set_last_error(const std::string& m);
}

namespace {

int fail(int code, const std::string& m) {
  gsbn::set_last_error(m);
  return code;
}

/* E = beta E + 0: the epilogue of the product when no row is active */
__global__ void re_decay(float* E, int64_t n, float beta) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    E[i] = beta * E[i] + 0.0f;
}

}  // namespace

struct gsbn_recall {
  gsbn_recall_desc d;
  int N = 0, Kp = 0, Np = 0, Bp = 0, W = 0, dmin = 1, dmax = 0, delay = 0;
  int R = 0, L = 0;
  bool wave = false; /* recall_wave_kernel covers this population */
  DBuf<float> dsup, epsc, bj, wij;
  DBuf<int32_t> count, di, inv_off, inv_slot, spk_cnt, out_idx, out_cnt, one, src_cnt;
  DBuf<uint16_t> spk_list, S, WT, Wb, src_list;
  DBuf<int16_t> clamp;
  DBuf<float> wmask;
  DBuf<int8_t> raster;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  ~gsbn_recall() {
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

extern "C" {

int gsbn_spike_gemm(int32_t B, int32_t N, int32_t Kp, const uint16_t* S, const uint16_t* WT,
                    float* E, float beta, void* stream) {
  if (B <= 0 || N <= 0 || Kp <= 0 || Kp % GM_BK || !S || !WT || !E) return GSBN_ERR_ARG;
  auto launch = [&](auto kernel, int bm, int threads) {
    const int mtiles = (B + bm - 1) / bm, ntiles = (N + bm - 1) / bm;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(mtiles * (int64_t)ntiles)), dim3(threads), 0,
                       (hipStream_t)stream, S, WT, E, B, N, Kp, beta, mtiles, ntiles);
  };
  const int64_t tiles = (int64_t)((B + GM_BM - 1) / GM_BM) * ((N + GM_BN - 1) / GM_BN);
  if (tiles > 0x7fffffff) return GSBN_ERR_UNSUPPORTED;
  if (tiles < GM_SMALL) launch(spike_gemm_kernel<64, 64, 2, 2>, 64, 256);
  else launch(spike_gemm_kernel<GM_BM, GM_BN, 2, 4>, GM_BM, 512);
  return ret(hipGetLastError());
}

gsbn_recall* gsbn_recall_new(const gsbn_recall_desc* d) {
  if (!d || d->H <= 0 || d->M <= 0 || d->M > RE_THREADS_MAX || d->C <= 0 || d->batch <= 0 ||
      d->batch > 65535 ||
      !d->ii || !d->di || !d->wij || !d->bj ||
      (d->mode != GSBN_RECALL_EXACT && d->mode != GSBN_RECALL_MFMA)) {
    fail(GSBN_ERR_ARG, "gsbn_recall_new: invalid description");
    return nullptr;
  }
  gsbn_recall* r = new gsbn_recall();
  r->d = *d;
  r->d.ii = nullptr;
  r->d.di = nullptr;
  r->d.wij = nullptr;
  r->d.bj = nullptr;
  const int H = d->H, M = d->M, C = d->C, B = d->batch;
  const int N = H * M;
  const int64_t R = (int64_t)H * C;
  r->N = N;
  r->W = (C + 31) / 32;
  auto bad = [&](int code, const std::string& m) -> gsbn_recall* {
    fail(code, m);
    delete r;
    return nullptr;
  };
  if ((size_t)r->W * 4 > 48 * 1024) return bad(GSBN_ERR_UNSUPPORTED, "gsbn_recall_new: C too large");
  /* delays and the inverse connectivity per (HCU, source unit) */
  std::vector<int32_t> off((size_t)H * (N + 1), 0), slots;
  int dmin = 32, dmax = 0;
  for (int h = 0; h < H; ++h) {
    std::vector<int32_t> cnt(N, 0);
    for (int k = 0; k < C; ++k) {
      const int s = d->ii[(int64_t)h * C + k];
      if (s < 0) continue;
      if (s >= N) return bad(GSBN_ERR_ARG, "gsbn_recall_new: ii out of range");
      const int dl = d->di[(int64_t)h * C + k];
      if (dl < 1 || dl > 31) return bad(GSBN_ERR_ARG, "gsbn_recall_new: delay outside [1, 31]");
      cnt[s]++;
      dmin = std::min(dmin, dl);
      dmax = std::max(dmax, dl);
    }
    int32_t* o = off.data() + (size_t)h * (N + 1);
    o[0] = (int32_t)slots.size();
    for (int s = 0; s < N; ++s) o[s + 1] = o[s] + cnt[s];
    slots.resize((size_t)o[N]);
    std::vector<int32_t> fill(o, o + N);
    for (int k = 0; k < C; ++k) {
      const int s = d->ii[(int64_t)h * C + k];
      if (s >= 0) slots[(size_t)fill[s]++] = k;
    }
  }
  if (dmax == 0) {
    dmin = 1;
    dmax = 0;
  }
  r->dmin = dmin;
  r->dmax = dmax;
  if (d->mode == GSBN_RECALL_MFMA && dmax > 0 && dmin != dmax)
    return bad(GSBN_ERR_UNSUPPORTED, "gsbn_recall_new: the mfma support needs one delay for all rows");
  r->delay = dmax;
  if (slots.empty()) slots.push_back(0);
  hipError_t e = hipSuccess;
  auto ok = [&](hipError_t x) {
    if (e == hipSuccess) e = x;
  };
  const int64_t BN = (int64_t)B * N;
  ok(r->dsup.alloc((size_t)BN));
  ok(r->epsc.alloc((size_t)BN));
  ok(r->count.alloc((size_t)BN));
  ok(r->bj.upload(d->bj, (size_t)N));
  ok(r->out_idx.alloc((size_t)B * H));
  ok(r->out_cnt.alloc((size_t)B * H));
  ok(r->clamp.alloc((size_t)B * H));
  ok(r->wmask.alloc((size_t)B * H));
  /* one wave per (HCU, cue) up to 256 units and 65536 sources (its lists hold
   * 16-bit units); the workgroup-per-pair kernels take larger populations */
  r->wave = M <= 256 && N <= 65536;
  r->L = std::min(dmin + 2, 8);
  r->R = std::max(dmax, dmin) + 2 + 2 * r->L;
  if (d->mode == GSBN_RECALL_EXACT) {
    ok(r->wij.upload(d->wij, (size_t)(R * M)));
    ok(r->di.upload(d->di, (size_t)R));
    ok(r->inv_off.upload(off.data(), off.size()));
    ok(r->inv_slot.upload(slots.data(), slots.size()));
    if (r->wave) {
      ok(r->one.alloc((size_t)H * N));
      if (e == hipSuccess) {
        hipLaunchKernelGGL(recall_one_kernel, dim3(grid_of((int64_t)H * N)), dim3(256), 0, 0,
                           (int64_t)H * N, N, r->inv_off.p, r->inv_slot.p, r->one.p);
        ok(hipGetLastError());
        ok(hipStreamSynchronize(0)); /* the runs have a stream of their own */
      }
    } else {
      ok(r->spk_cnt.alloc((size_t)RE_RING * B * H));
      ok(r->spk_list.alloc((size_t)RE_RING * B * N));
    }
  } else {
    /* dense W in bf16, by destination unit (WT, for the product) and by
     * source (Wb, for the wave kernel), from the slots of each source */
    r->Kp = (N + GM_BK - 1) / GM_BK * GM_BK;
    r->Np = (N + GM_BN - 1) / GM_BN * GM_BN;
    r->Bp = (B + GM_BM - 1) / GM_BM * GM_BM;
    /* The dense product costs 2 M N flops per pair and step whatever spikes;
     * the wave kernel only its population step and the active rows.  Measured
     * per pair and step, product with its population step against the wave
     * kernel: 3.0 / 1.6 ns at 100 x 100 (8192 cues), 3.3 / 1.7 at 40 x 128,
     * 0.72 / 0.80 at 60 x 20 and 0.81 / 0.89 at 180 x 12, where the product
     * is small and the leaner population step of its path wins: the line is
     * at M N = 60000.  Below it small batches still gain, because the wave
     * kernel takes L steps per launch instead of two launches per step
     * (about 4 us a step, 0.1 ns for each of 40000 pairs).  The rates hold up
     * to one active source per two hypercolumns and step (6.06 ms for 20
     * steps of 2048 cues at maxfq dt = 0.5 against 5.86 at 0.1); a
     * hypercolumn's activities sum to at most 1, so maxfq dt bounds them. */
    if (!(d->maxfqdt <= 0.5f) ||
        ((int64_t)M * N < 60000 && (int64_t)B * H >= 40000))
      r->wave = false;
    DBuf<float> w;
    DBuf<int32_t> o, sl, bad;
    const int32_t zero = 0;
    ok(w.upload(d->wij, (size_t)(R * M)));
    ok(o.upload(off.data(), off.size()));
    ok(sl.upload(slots.data(), slots.size()));
    ok(bad.upload(&zero, 1));
    if (r->wave) ok(r->Wb.alloc((size_t)H * N * M));
    ok(r->WT.alloc((size_t)r->Np * r->Kp));
    if (e == hipSuccess) {
      const int64_t nw = (int64_t)r->Np * r->Kp / 2;
      hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(nw)), dim3(256), 0, 0,
                         reinterpret_cast<float*>(r->WT.p), nw, 0.0f);
      hipLaunchKernelGGL(recall_weights_kernel, dim3(N, std::min(H, 65535)), dim3(M <= 64 ? 64 : 128), 0, 0, H, M, C, N,
                         r->Kp, w.p, o.p, sl.p, r->Wb.p, r->WT.p, bad.p);
      ok(hipGetLastError());
      int32_t nonfinite = 0;
      ok(hipMemcpy(&nonfinite, bad.p, sizeof(nonfinite), hipMemcpyDeviceToHost));
      /* an infinite or NaN weight reaches every cue through the product's
       * zeros; only the dense product has that */
      if (nonfinite) r->wave = false;
    }
  }
  if (r->wave) {
    ok(r->src_cnt.alloc((size_t)r->R * B));
    ok(r->src_list.alloc((size_t)r->R * B * N));
  } else if (d->mode == GSBN_RECALL_MFMA) {
    /* the spike matrices of the product (a handle of the wave kernel makes
     * them in its first run that asks for the product's time) */
    ok(r->S.alloc((size_t)RE_RING * r->Bp * r->Kp));
  }
  ok(hipStreamCreateWithFlags(&r->stream, hipStreamNonBlocking));
  ok(hipEventCreate(&r->ev0));
  ok(hipEventCreate(&r->ev1));
  if (e != hipSuccess) return bad((int)e, std::string("gsbn_recall_new: ") + hipGetErrorString(e));
  return r;
}

void gsbn_recall_free(gsbn_recall* r) { delete r; }

}  // extern "C"

namespace {

/* the run by recall_wave_kernel, L steps per launch */
int run_wave(gsbn_recall* r, ReArgs a, int steps, int8_t* raster) {
  hipStream_t s = r->stream;
  const gsbn_recall_desc& d = r->d;
  const int B = d.batch;
  const int64_t BN = (int64_t)B * r->N, nc = (int64_t)r->R * B;
  hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(nc)), dim3(256), 0, s,
                     reinterpret_cast<float*>(r->src_cnt.p), nc, 0.0f);
  /* raster steps kept on the device before a copy to the host */
  int64_t keep = 0;
  if (raster) {
    keep = std::min<int64_t>(steps, std::max<int64_t>(1, ((int64_t)256 << 20) / BN));
    if ((int64_t)r->raster.n < keep * BN) {
      const hipError_t e = r->raster.alloc((size_t)(keep * BN));
      if (e != hipSuccess) return fail((int)e, "gsbn_recall_run: raster buffer");
    }
    a.raster = r->raster.p;
  }
  a.raster_t0 = 1;
  const int upl = (d.M + 63) / 64;
  const dim3 grid((unsigned)(8 * ((d.H + 7) / 8) * ((B + RW_WAVES - 1) / RW_WAVES)));
  const dim3 block(64 * RW_WAVES);
  const bool bf = d.mode == GSBN_RECALL_MFMA;
  for (int t = 1; t <= steps;) {
    int nt = std::min(r->L, steps - t + 1);
    if (raster) nt = (int)std::min<int64_t>(nt, a.raster_t0 + keep - t);
    const int last = t + nt > steps ? 1 : 0;
#define RW_LAUNCH(U, F) \
  hipLaunchKernelGGL((recall_wave_kernel<U, F>), grid, block, 0, s, a, t, nt, last)
    if (upl == 1) {
      if (bf) RW_LAUNCH(1, true);
      else RW_LAUNCH(1, false);
    } else if (upl == 2) {
      if (bf) RW_LAUNCH(2, true);
      else RW_LAUNCH(2, false);
    } else {
      if (bf) RW_LAUNCH(4, true);
      else RW_LAUNCH(4, false);
    }
#undef RW_LAUNCH
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail((int)e, "recall_wave_kernel");
    t += nt;
    if (raster && (t > steps || t == a.raster_t0 + keep)) {
      e = hipMemcpyAsync(raster + (int64_t)(a.raster_t0 - 1) * BN, r->raster.p,
                         (size_t)((t - a.raster_t0) * BN), hipMemcpyDeviceToHost, s);
      if (e != hipSuccess) return fail((int)e, "gsbn_recall_run: raster");
      a.raster_t0 = t;
    }
  }
  return 0;
}

}  // namespace

extern "C" {

int gsbn_recall_run(gsbn_recall* r, const int16_t* clamp, const float* wmask, int32_t steps,
                    int32_t count_from, int32_t* out_idx, int32_t* out_cnt, int8_t* raster,
                    double* support_ms) {
  if (!r || !clamp || !wmask || steps < 0 || !out_idx || !out_cnt)
    return fail(GSBN_ERR_ARG, "gsbn_recall_run: invalid arguments");
  const gsbn_recall_desc& d = r->d;
  const int B = d.batch, H = d.H, M = d.M, N = r->N;
  const int64_t BN = (int64_t)B * N;
  hipStream_t s = r->stream;
  hipError_t e = hipMemcpyAsync(r->clamp.p, clamp, (size_t)B * H * 2, hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(r->wmask.p, wmask, (size_t)B * H * 4, hipMemcpyHostToDevice, s);
  if (e != hipSuccess) return fail((int)e, "gsbn_recall_run: upload");
  /* the product's time is wanted: one product per step, as below */
  const bool wave = r->wave && steps > 0 && !(support_ms && d.mode == GSBN_RECALL_MFMA);
  /* initial state: dsup = log(1/M) (Pop.cpp:59), E = 0, counts 0, empty queue */
  const float dsup0 = (float)log(1.0 / M);
  if (!wave) {
    hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(BN)), dim3(256), 0, s, r->dsup.p, BN, dsup0);
    hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(BN)), dim3(256), 0, s, r->epsc.p, BN, 0.0f);
    hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(BN)), dim3(256), 0, s,
                       reinterpret_cast<float*>(r->count.p), BN, 0.0f);
    if (d.mode == GSBN_RECALL_EXACT) {
      if (!r->spk_cnt.p) {
        /* no steps: the lists are not used */
      } else {
        const int64_t nc = (int64_t)RE_RING * B * H;
        hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(nc)), dim3(256), 0, s,
                           reinterpret_cast<float*>(r->spk_cnt.p), nc, 0.0f);
      }
    } else {
      const int64_t ns = (int64_t)RE_RING * r->Bp * r->Kp;
      if (!r->S.p && steps > 0 && (e = r->S.alloc((size_t)ns)) != hipSuccess)
        return fail((int)e, "gsbn_recall_run: spike matrices");
      if (steps > 0)
        hipLaunchKernelGGL(re_fill_f32, dim3(grid_of(ns / 2)), dim3(256), 0, s,
                           reinterpret_cast<float*>(r->S.p), ns / 2, 0.0f);
    }
    if (raster && (int64_t)r->raster.n < BN) {
      e = r->raster.alloc((size_t)BN);
      if (e != hipSuccess) return fail((int)e, "gsbn_recall_run: raster buffer");
    }
  }
  ReArgs a;
  memset(&a, 0, sizeof(a));
  a.B = B;
  a.Bp = r->Bp;
  a.H = H;
  a.M = M;
  a.C = d.C;
  a.N = N;
  a.Kp = r->Kp;
  a.W = r->W;
  a.dmin = r->dmin;
  a.dmax = r->dmax;
  a.count_from = count_from;
  a.mode = d.mode;
  a.seed = d.seed;
  a.taumdt = d.taumdt;
  a.wtagain = d.wtagain;
  a.maxfqdt = d.maxfqdt;
  a.igain = d.igain;
  a.wgain = d.wgain;
  a.lgbias = d.lgbias;
  a.snoise = d.snoise;
  a.kepsc = d.kepsc;
  a.lg_on = d.lg_on;
  a.lg_off = d.lg_off;
  a.dsup = r->dsup.p;
  a.epsc = r->epsc.p;
  a.count = r->count.p;
  a.bj = r->bj.p;
  a.wij = r->wij.p;
  a.di = r->di.p;
  a.inv_off = r->inv_off.p;
  a.inv_slot = r->inv_slot.p;
  a.spk_cnt = r->spk_cnt.p;
  a.spk_list = r->spk_list.p;
  a.S = r->S.p;
  a.clamp = r->clamp.p;
  a.wmask = r->wmask.p;
  a.raster = raster ? r->raster.p : nullptr;
  a.R = r->R;
  a.L = r->L;
  a.Np = r->Np;
  a.dsup0 = dsup0;
  a.one = r->one.p;
  a.Wb = r->Wb.p;
  a.WT = r->WT.p;
  a.src_cnt = r->src_cnt.p;
  a.src_list = r->src_list.p;
  a.out_idx = r->out_idx.p;
  a.out_cnt = r->out_cnt.p;
  if (wave) {
    const int rc = run_wave(r, a, steps, raster);
    if (rc) return rc;
  }
  const int threads = ((M + 63) / 64) * 64;
  const size_t lds = d.mode == GSBN_RECALL_EXACT ? ((size_t)r->W + RE_ROWS_MAX) * 4 : 0;
  const float beta = 1 - d.kepsc;
  double gemm_ms = 0.0;
  /* the mfma mode's population step: one wave per (HCU, cue) up to 256 units */
  const int upl = (M + 63) / 64;
  const bool wave_step = d.mode == GSBN_RECALL_MFMA && upl <= 4;
  const unsigned wave_grid = (unsigned)(((int64_t)B * H + 3) / 4);
  for (int t = 1; !wave && t <= steps; ++t) {
    if (wave_step) {
      if (upl == 1)
        hipLaunchKernelGGL(recall_pop_wave_kernel<1>, dim3(wave_grid), dim3(256), 0, s, a, t);
      else if (upl == 2)
        hipLaunchKernelGGL(recall_pop_wave_kernel<2>, dim3(wave_grid), dim3(256), 0, s, a, t);
      else
        hipLaunchKernelGGL(recall_pop_wave_kernel<4>, dim3(wave_grid), dim3(256), 0, s, a, t);
    } else {
      hipLaunchKernelGGL(recall_step_kernel, dim3(H, B), dim3(threads), lds, s, a, t);
    }
    if ((e = hipGetLastError()) != hipSuccess) return fail((int)e, "recall_step_kernel");
    if (d.mode == GSBN_RECALL_MFMA) {
      const int src = t - r->delay - 2;
      if (support_ms) (void)hipEventRecord(r->ev0, s);
      if (src >= 1 && r->delay > 0) {
        const uint16_t* Sp = r->S.p + (int64_t)(src % RE_RING) * r->Bp * r->Kp;
        int rc = gsbn_spike_gemm(B, N, r->Kp, Sp, r->WT.p, r->epsc.p, beta, s);
        if (rc) return fail(rc, "gsbn_spike_gemm");
      } else {
        /* no row can be active yet: the decay alone */
        hipLaunchKernelGGL(re_decay, dim3(grid_of(BN)), dim3(256), 0, s, r->epsc.p, BN, beta);
        if ((e = hipGetLastError()) != hipSuccess) return fail((int)e, "re_decay");
      }
      if (support_ms) {
        (void)hipEventRecord(r->ev1, s);
        (void)hipEventSynchronize(r->ev1);
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, r->ev0, r->ev1);
        gemm_ms += ms;
      }
    }
    if (raster) {
      e = hipMemcpyAsync(raster + (int64_t)(t - 1) * BN, r->raster.p, (size_t)BN,
                         hipMemcpyDeviceToHost, s);
      if (e != hipSuccess) return fail((int)e, "gsbn_recall_run: raster");
    }
  }
  const int64_t BH = (int64_t)B * H;
  if (!wave)
    hipLaunchKernelGGL(recall_argmax_kernel, dim3(grid_of(BH)), dim3(256), 0, s, B, H, M,
                       r->count.p, r->out_idx.p, r->out_cnt.p);
  e = hipMemcpyAsync(out_idx, r->out_idx.p, (size_t)BH * 4, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(out_cnt, r->out_cnt.p, (size_t)BH * 4, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return fail((int)e, std::string("gsbn_recall_run: ") + hipGetErrorString(e));
  if (support_ms) *support_ms = gemm_ms;
  return 0;
}

}  // extern "C"
