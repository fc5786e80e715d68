// Row-count-invariant log-softmax + target gather over a fixed-leaf exp-sum tree.
//
// Function computed per row (the expression tree of the reference's leaf_sum_exp /
// finalize_rows / full_row_logprobs, skyrl/backends/skyrl_train/isoexec/ops/logprobs/rowinv.py:136-245):
//   m      = max_j x[j]                                   (exact, order-free)
//   leaf_g = Kahan-fp32 sum over blocks b of  blocksum(g, b)      g = 0..G-1, L = V/G columns each
//   S      = balanced pairwise fold of the G leaves               (combine_order(G))
//   logp   = (x[target] - m) - log(S)        lse = m + log(S)
// blocksum(g, b) covers BLOCK = 4096 consecutive columns of leaf g (the last block masked):
//   column sums col[p] = sum over the 8 chunks c of term[c*512 + p], left to right, p = 0..511,
//   then the adjacent-pairwise tree over the 512 columns,
//   term[i] = exp2((x[i] - m) * log2(e)) for live columns and 0 for masked ones.
// Every quantity above depends only on (V, G) and the row's own values, never on the number
// of rows or on which launch shape ran, so a row's bits are the same at any row count.
//
// Two launch shapes evaluate that same function:
//   * rows >= IX_LP_SPLIT_BELOW : one 512-thread workgroup per row, one launch (wide rows: a workgroup per CU that keeps them);
//   * fewer rows                : row split over many workgroups (partial max, block sums,
//                                 finalize) so a single decode row still fills the chip.
#include "ix_common.h"
#include "../../include/isoexec_hip.h"

#define IX_LP_BLOCK 4096
#define IX_LP_MAX_UNITS 4096  // G * ceil(L / BLOCK) a workgroup can hold in LDS
#define IX_LP_MAX_G 64
#define IX_LP_SPLIT_BELOW 192
#define IX_LP_SEG 8192  // columns per partial-max / full-row-write workgroup in the split shape

// One wave sums one block. `blk` points at the block's first column, n_valid <= 4096 columns
// exist. Returns the block sum in every lane.
// `row_max()` yields the row maximum; it is called after the block's loads are issued, so a maximum that is itself
// read from memory does not put its latency in front of theirs.
template <typename T, typename MaxFn>
__device__ __forceinline__ float ix_block_expsum_with(const T* __restrict__ blk, int n_valid, const MaxFn& row_max,
                                                      bool vec, int lane) {
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (vec) {
    // vec implies that the leaf length is a multiple of 8, so a group of 8 columns is whole or absent. All eight
    // groups are requested before the first is used: a lane has eight independent loads in flight instead of one
    // (a load, its wait and its sum per group is bound by memory latency). An absent group reads the block's first
    // columns instead (no branch between the loads) and adds +0.0. The sums are the ones below: slot i adds its
    // groups in ascending c.
    IxRaw8<T> raw[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int off = c * 512 + lane * 8;
      raw[c].load(blk + ((n_valid - off >= 8) ? off : 0));
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads are issued back to back; widening waits with the sums
    const float m = row_max();
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const bool whole = n_valid - (c * 512 + lane * 8) >= 8;
      float x[8];
      raw[c].widen(x);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = acc[i] + (whole ? ix_exp_fast(x[i] - m) : 0.0f);
    }
    return ix_lane_tree<64>(ix_tree8(acc));
  }
  const float m = row_max();
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int off = c * 512 + lane * 8;
    const int valid = n_valid - off;
    if (valid > 0) {  // a fully masked group adds +0.0 to every slot: a no-op on the bits
      float x[8];
      ix_load8(blk + off, valid, vec, 0.0f, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float t = (i < valid) ? ix_exp_fast(x[i] - m) : 0.0f;
        acc[i] = acc[i] + t;
      }
    }
  }
  return ix_lane_tree<64>(ix_tree8(acc));
}

template <typename T>
__device__ __forceinline__ float ix_block_expsum(const T* __restrict__ blk, int n_valid, float m, bool vec,
                                                 int lane) {
  return ix_block_expsum_with(blk, n_valid, [m]() { return m; }, vec, lane);
}

__device__ __forceinline__ float ix_kahan_blocks(const float* __restrict__ bsum, int nb) {
  float acc = 0.0f, comp = 0.0f;
  for (int b = 0; b < nb; ++b) {
    const float y = bsum[b] - comp;
    const float t = acc + y;
    comp = (t - acc) - y;
    acc = t;
  }
  return acc;
}

// In-place balanced fold; leaf[0] ends as the root. Stride doubling == combine_order(G) of
// skyrl/backends/skyrl_train/isoexec/ops/collectives/pik/plan.py:104-119.
__device__ __forceinline__ float ix_fold_leaves(float* leaf, int G) {
  for (int s = 1; s < G; s <<= 1)
    for (int i = 0; i + s < G; i += 2 * s) leaf[i] = leaf[i] + leaf[i + s];
  return leaf[0];
}

// log S of a row from its block sums, by one wave: a lane per leaf, folded as ix_fold_leaves does. Valid in lane 0.
__device__ __forceinline__ float ix_log_total(const float* __restrict__ bsum, int G, int NB, int lane) {
  float leaf = lane < G ? ix_kahan_blocks(bsum + lane * NB, NB) : 0.0f;
  for (int s = 1; s < G; s <<= 1) leaf = leaf + __shfl_xor(leaf, s, IX_WAVE);
  return ix_log(leaf);
}

template <typename T>
__device__ __forceinline__ void ix_lp_emit(const T* __restrict__ xr, int V, float m, float log_s,
                                           const int64_t* __restrict__ target, long row, float* out_lp,
                                           float* out_lse) {
  if (out_lp) {
    const int64_t t = target[row];
    const bool valid = (t >= 0) && (t < (int64_t)V);
    float sampled = 0.0f;
    if (valid) {
      float o[8];
      ix_load8(xr + t, 1, false, 0.0f, o);
      sampled = o[0];
    }
    out_lp[row] = valid ? (sampled - m) - log_s : 0.0f;
  }
  if (out_lse) out_lse[row] = m + log_s;
}

// ---------------------------------------------------------------------------------------------
// Shape 1: one workgroup (8 waves) per row.
template <typename T>
__global__ __launch_bounds__(512) void k_lp_row(const T* __restrict__ x, long row_stride, int V, int G,
                                                const int64_t* __restrict__ target, float* __restrict__ out_lp,
                                                float* __restrict__ out_lse, float* __restrict__ out_full,
                                                long full_stride, int vec) {
  constexpr int NT = 512, NW = NT / 64;
  __shared__ float s_wmax[NW];
  __shared__ float s_bsum[IX_LP_MAX_UNITS];
  __shared__ float s_leaf[IX_LP_MAX_G];
  __shared__ float s_fin[2];
  const long row = blockIdx.x;
  const T* xr = x + row * row_stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int L = V / G;
  const int NB = (L + IX_LP_BLOCK - 1) / IX_LP_BLOCK;

  float m = IX_NEG_INF;
  // The maximum's pass. V % 8 == 0 under vec: whole groups, four of them requested before the first is used ([1000, 151936]:
  // fp32 182 -> 176 us, bf16 93 -> 88 for the whole kernel, 6.9 TB/s over the row's two readings; neither more threads
  // per row nor fewer rows in flight, so that the second reading would come from the memory-side cache, moved it).
  if (vec) {
    for (int off0 = tid * 8; off0 < V; off0 += NT * 32) {
      IxRaw8<T> raw[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int off = off0 + c * NT * 8;
        raw[c].load(xr + (off < V ? off : off0));
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float o[8];
        raw[c].widen(o);
        m = fmaxf(m, ix_tree8_max(o));
      }
    }
  } else {
    for (long off = (long)tid * 8; off < V; off += NT * 8) {
      float o[8];
      ix_load8(xr + off, V - off, false, IX_NEG_INF, o);
      m = fmaxf(m, ix_tree8_max(o));
    }
  }
  m = ix_lane_max<64>(m);
  if (lane == 0) s_wmax[wave] = m;
  __syncthreads();
  m = s_wmax[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) m = fmaxf(m, s_wmax[w]);

  const int units = G * NB;
  for (int u = wave; u < units; u += NW) {
    const int g = u / NB, b = u - g * NB;
    const long base = (long)g * L + (long)b * IX_LP_BLOCK;
    const int nv = min(IX_LP_BLOCK, L - b * IX_LP_BLOCK);
    const float bs = ix_block_expsum(xr + base, nv, m, vec != 0, lane);
    if (lane == 0) s_bsum[u] = bs;
  }
  __syncthreads();
  if (tid < G) s_leaf[tid] = ix_kahan_blocks(s_bsum + tid * NB, NB);
  __syncthreads();
  if (tid == 0) {
    const float S = ix_fold_leaves(s_leaf, G);
    const float log_s = ix_log(S);
    s_fin[0] = m;
    s_fin[1] = log_s;
    ix_lp_emit(xr, V, m, log_s, target, row, out_lp, out_lse);
  }
  if (out_full) {
    __syncthreads();
    const float mm = s_fin[0], ls = s_fin[1];
    float* orow = out_full + row * full_stride;
    for (long off = (long)tid * 8; off < V; off += NT * 8) {
      float o[8];
      ix_load8(xr + off, V - off, vec != 0, 0.0f, o);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (off + i < V) orow[off + i] = (o[i] - mm) - ls;
    }
  }
}

// Shape 1 with the row kept on the CU between the maximum and the sums. A workgroup per CU walks the rows; a wave keeps HU of its
// blocks in registers and LU in LDS, reads the others twice, and asks for the next row's block as soon as this row's is summed.
// The blocks, their sums and the fold are k_lp_row's. Bound by HBM: of [1000, 151936] in bf16 all 40 blocks stay (5 a wave, 160
// registers), 93 -> 70 us; in fp32 24 (two a wave in registers, one in LDS), 181 -> 129; 2900 rows 259 -> 179 and 506 -> 354.
// Three fp32 blocks in registers leave none to work with (spilled loads have to be waited for: 155).
// The registers as they are: no widened copy of them lives on from an earlier use.
__device__ __forceinline__ void ix_lp_keep(IxRaw8<bf16_t>& r) {
  asm volatile("" : "+v"(r.v.x), "+v"(r.v.y), "+v"(r.v.z), "+v"(r.v.w));
}
__device__ __forceinline__ void ix_lp_keep(IxRaw8<float>&) {}
#define IX_LP_HELD_UNITS 512
template <typename T, int HU, int LU>
__global__ __launch_bounds__(512) void k_lp_row_held(const T* __restrict__ x, long row_stride, long rows, int V, int G,
                                                     const int64_t* __restrict__ target, float* __restrict__ out_lp,
                                                     float* __restrict__ out_lse) {
  constexpr int NW = 8, CH = 4;  // CH: groups of a block that is not kept requested at once
  extern __shared__ __align__(16) char ix_lp_lds[];
  __shared__ float s_wmax[2][NW];
  __shared__ float s_bsum[2][IX_LP_HELD_UNITS];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar, and the blocks' addresses with it
  const int L = V / G;
  const int NB = (L + IX_LP_BLOCK - 1) / IX_LP_BLOCK;
  const int units = G * NB;
  IxRaw8<T>* kept = reinterpret_cast<IxRaw8<T>*>(ix_lp_lds) + (size_t)wave * LU * 8 * 64 + lane;  // [LU][8] of this lane

  unsigned lane8 = lane * 8;
  auto width = [&](int u) __attribute__((always_inline)) { return min(IX_LP_BLOCK, L - u % NB * IX_LP_BLOCK); };
  // group c of block u; one past the block's end reads its first columns instead, which changes no maximum
  auto load = [&](IxRaw8<T>& r, const T* xr, int u, int c) __attribute__((always_inline)) {
    const T* blk = xr + (long)(u / NB) * L + u % NB * IX_LP_BLOCK;
    const unsigned off = c * 512 + lane8;
    r.load(blk + (off + 8 <= (unsigned)width(u) ? off : 0u));
  };
  auto add = [&](float (&acc)[8], const IxRaw8<T>& r, float m, int u, int c) __attribute__((always_inline)) {
    // The term of a group past the end is exp(v - inf) = +0, or a NaN if v is one or +inf: v is a column of this block then,
    // whose own term is a NaN as well.
    const float mm = (unsigned)(c * 512) + lane8 + 8 <= (unsigned)width(u) ? m : -IX_NEG_INF;
    float v[8];
    r.widen(v);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = acc[i] + ix_exp_fast(v[i] - mm);
  };

  IxRaw8<T> held[HU][8];
  long row = blockIdx.x;
#pragma unroll
  for (int j = 0; j < HU; ++j) {
    if (wave + NW * j < units) {
#pragma unroll
      for (int c = 0; c < 8; ++c) load(held[j][c], x + row * row_stride, wave + NW * j, c);
    }
  }
  for (int par = 0; row < rows; row += gridDim.x, par ^= 1) {
    const T* xr = x + row * row_stride;
    float m = IX_NEG_INF;
    asm volatile("" : "+v"(lane8));  // the groups' offsets are computed where they are used, not kept in registers from row to row
    for (int u = wave + NW * HU; u < units; u += NW) {
      const int l = (u - wave) / NW - HU;
#pragma unroll
      for (int c0 = 0; c0 < 8; c0 += CH) {
        IxRaw8<T> raw[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) load(raw[c], xr, u, c0 + c);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          float v[8];
          raw[c].widen(v);
          m = fmaxf(m, ix_tree8_max(v));
          if (LU > 0 && l < LU) kept[(l * 8 + c0 + c) * 64] = raw[c];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < HU; ++j) {
      if (wave + NW * j < units) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          float v[8];
          held[j][c].widen(v);
          m = fmaxf(m, ix_tree8_max(v));
        }
      }
    }
    m = ix_lane_max<64>(m);
    if (lane == 0) s_wmax[par][wave] = m;
    __syncthreads();
    m = s_wmax[par][0];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, s_wmax[par][w]);

#pragma unroll
    for (int j = 0; j < HU; ++j)
#pragma unroll
      for (int c = 0; c < 8; ++c) ix_lp_keep(held[j][c]);
    const long next = row + gridDim.x;
    asm volatile("" : "+v"(lane8));
#pragma unroll
    for (int j = 0; j < HU; ++j) {
      const int u = wave + NW * j;
      if (u < units) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 8; ++c) add(acc, held[j][c], m, u, c);
        if (next < rows) {
#pragma unroll
          for (int c = 0; c < 8; ++c) load(held[j][c], x + next * row_stride, u, c);
        }
        const float bs = ix_lane_tree<64>(ix_tree8(acc));
        if (lane == 0) s_bsum[par][u] = bs;
      }
    }
    for (int u = wave + NW * HU; u < units; u += NW) {
      const int l = (u - wave) / NW - HU;
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c0 = 0; c0 < 8; c0 += CH) {
        IxRaw8<T> raw[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          if (LU > 0 && l < LU) raw[c] = kept[(l * 8 + c0 + c) * 64];
          else load(raw[c], xr, u, c0 + c);
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) add(acc, raw[c], m, u, c0 + c);
      }
      const float bs = ix_lane_tree<64>(ix_tree8(acc));
      if (lane == 0) s_bsum[par][u] = bs;
    }
    __syncthreads();
    if (wave == 0) {  // the others go on with the next row: its maxima and sums have places of their own
      const float log_s = ix_log_total(s_bsum[par], G, NB, lane);
      if (lane == 0) ix_lp_emit(xr, V, m, log_s, target, row, out_lp, out_lse);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Shape 2: the row split over many workgroups. Workspace layout (floats):
//   pmax [rows, P]  P = ceil(V / IX_LP_SEG)
//   bsum [rows, U]  U = G * NB
//   fin  [rows, 2]  (m, log S), for full rows of many blocks a leaf
template <typename T>
__global__ __launch_bounds__(256) void k_lp_partmax(const T* __restrict__ x, long row_stride, int V, int P,
                                                    float* __restrict__ pmax, int vec) {
  __shared__ float s_w[4];
  const long row = blockIdx.x / P;  // parts fastest: consecutive workgroups read consecutive memory
  const int p = blockIdx.x % P;
  const T* xr = x + row * row_stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long lo = (long)p * IX_LP_SEG;
  const long hi = min((long)V, lo + IX_LP_SEG);
  float m = IX_NEG_INF;
  for (long off = lo + (long)tid * 8; off < hi; off += 256 * 8) {
    float o[8];
    ix_load8(xr + off, hi - off, vec != 0, IX_NEG_INF, o);
    m = fmaxf(m, ix_tree8_max(o));
  }
  m = ix_lane_max<64>(m);
  if (lane == 0) s_w[wave] = m;
  __syncthreads();
  if (tid == 0) pmax[row * P + p] = fmaxf(fmaxf(s_w[0], s_w[1]), fmaxf(s_w[2], s_w[3]));
}

__device__ __forceinline__ float ix_row_max_from_parts(const float* __restrict__ pm, int P, int lane) {
  float m = IX_NEG_INF;
  for (int i = lane; i < P; i += 64) m = fmaxf(m, pm[i]);
  return ix_lane_max<64>(m);
}

// Work order: (row, group of 4 units) with the units fastest, i.e. memory order, walked in 8 XCD runs
// (ix_xcd_run_position). On 4096 x 151936 bf16: rows fastest 0.234 ms, memory order 0.219 ms, XCD runs 0.210 ms.
template <typename T>
__global__ __launch_bounds__(256) void k_lp_blocksums(const T* __restrict__ x, long row_stride, int V, int G,
                                                      int P, const float* __restrict__ pmax,
                                                      float* __restrict__ bsum, int vec, int ny,
                                                      unsigned total) {
  unsigned l;
  if (!ix_xcd_run_position(blockIdx.x, total, &l)) return;
  const long row = l / ny;
  const int by = l % ny;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int L = V / G;
  const int NB = (L + IX_LP_BLOCK - 1) / IX_LP_BLOCK;
  const int units = G * NB;
  const int u = by * 4 + wave;
  if (u >= units) return;
  const int g = u / NB, b = u - g * NB;
  const long base = (long)g * L + (long)b * IX_LP_BLOCK;
  const int nv = min(IX_LP_BLOCK, L - b * IX_LP_BLOCK);
  const float bs = ix_block_expsum_with(
      x + row * row_stride + base, nv, [&]() { return ix_row_max_from_parts(pmax + row * P, P, lane); }, vec != 0, lane);
  if (lane == 0) bsum[row * units + u] = bs;
}

template <typename T>
__global__ __launch_bounds__(64) void k_lp_finalize(const T* __restrict__ x, long row_stride, int V, int G, int P,
                                                    const float* __restrict__ pmax,
                                                    const float* __restrict__ bsum, float* __restrict__ fin,
                                                    const int64_t* __restrict__ target,
                                                    float* __restrict__ out_lp, float* __restrict__ out_lse) {
  __shared__ float s_leaf[IX_LP_MAX_G];
  const long row = blockIdx.x;
  const int lane = threadIdx.x;
  const int L = V / G;
  const int NB = (L + IX_LP_BLOCK - 1) / IX_LP_BLOCK;
  const float m = ix_row_max_from_parts(pmax + row * P, P, lane);
  if (lane < G) s_leaf[lane] = ix_kahan_blocks(bsum + row * (long)(G * NB) + lane * NB, NB);
  __syncthreads();
  if (lane == 0) {
    const float S = ix_fold_leaves(s_leaf, G);
    const float log_s = ix_log(S);
    if (fin) {
      fin[row * 2] = m;
      fin[row * 2 + 1] = log_s;
    }
    ix_lp_emit(x + row * row_stride, V, m, log_s, target, row, out_lp, out_lse);
  }
}

// The whole row, and its lse. Every workgroup joins the row's block sums for itself (a wave, while the columns travel) instead
// of a launch in front that does it once: 4.6 us less for a decode step. Bound by HBM: four columns per lane and access, so that
// a store instruction is 1 KiB of the row, all of them requested first: 64 rows of 151936 26.5 -> 10.2 us (eight columns
// per lane stored one by one before). The join is a chain over a leaf's blocks, so with many of them the launch in front does it
// (fin). us joined everywhere / in front, bf16: 1 row of 192 blocks 24.4 / 25.0, 16 39.4 / 41.3, 64 117 / 97; of 256 29.5 / 29.1,
// 50.0 / 52.7, 171 / 136; of 384 40.4 / 39.1, 98 / 76, 332 / 209; 64 rows of 136 84 / 71, 16 of 2048 1417 / 442.
static bool ix_lp_joins_in_front(long rows, int NB) { return NB > 256 || (NB > 128 && rows >= 64); }
__device__ __forceinline__ void ix_lp_load4(const float* p, float (&v)[4]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void ix_lp_load4(const bf16_t* p, float (&v)[4]) {
  const uint2 a = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
  v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
}
template <typename T>
__global__ __launch_bounds__(256) void k_lp_fullwrite(const T* __restrict__ x, long row_stride, int V, int G, int P,
                                                      const float* __restrict__ pmax, const float* __restrict__ bsum,
                                                      const float* __restrict__ fin, float* __restrict__ out_full, long full_stride,
                                                      float* __restrict__ out_lse, int vec, int PW) {
  constexpr int GROUPS = IX_LP_SEG / (256 * 4);
  __shared__ float s_fin[2];
  const long row = blockIdx.x / PW;  // segments fastest
  const T* xr = x + row * row_stride;
  float* orow = out_full + row * full_stride;
  const int lo = (int)(blockIdx.x % PW) * IX_LP_SEG;
  const int hi = min(V, lo + IX_LP_SEG);
  float v[GROUPS][4];
  if (vec) {  // whole groups of four; an absent one reads the segment's first columns
#pragma unroll
    for (int c = 0; c < GROUPS; ++c) {
      const int off = lo + (c * 256 + (int)threadIdx.x) * 4;
      ix_lp_load4(xr + (off < hi ? off : lo), v[c]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (fin) {
    if (threadIdx.x < 2) s_fin[threadIdx.x] = fin[row * 2 + threadIdx.x];
  } else if (threadIdx.x < 64) {
    const int NB = (V / G + IX_LP_BLOCK - 1) / IX_LP_BLOCK;
    const float m = ix_row_max_from_parts(pmax + row * P, P, threadIdx.x);
    const float log_s = ix_log_total(bsum + row * (long)(G * NB), G, NB, threadIdx.x);
    if (threadIdx.x == 0) {
      s_fin[0] = m;
      s_fin[1] = log_s;
      if (out_lse && lo == 0) out_lse[row] = m + log_s;
    }
  }
  __syncthreads();
  const float mm = s_fin[0], ls = s_fin[1];
  if (vec) {
#pragma unroll
    for (int c = 0; c < GROUPS; ++c) {
      const int off = lo + (c * 256 + (int)threadIdx.x) * 4;
      if (off < hi)
        *reinterpret_cast<float4*>(orow + off) =
            make_float4((v[c][0] - mm) - ls, (v[c][1] - mm) - ls, (v[c][2] - mm) - ls, (v[c][3] - mm) - ls);
    }
    return;
  }
  for (int j = lo + (int)threadIdx.x; j < hi; j += 256) {
    float o[8];
    ix_load8(xr + j, 1, false, 0.0f, o);
    orow[j] = (o[0] - mm) - ls;
  }
}

// ---------------------------------------------------------------------------------------------
// Gradient of the sampled logprob (rowinv.py:573-612): grad[j] = -u * exp(x[j] - lse), plus u at the target, u = upstream[row]
// (0 for a target outside the vocabulary), rounded to the logits' type at the store. One pass: every logit is read once and
// every gradient written once. Bound by HBM: behind its forward, [1000, 151936] fp32 207 us with the default cache policy
// and 32 bytes per lane, 188 us = 6.5 TB/s past the caches with 16 (a non-temporal store has to fill whole lines by itself:
// 220 us with 32 bytes per lane); bf16 107 -> 106 and the forward behind it 109 -> 93. The same expression in elementwise
// passes took 600 us.
// A workgroup owns a segment of IX_LP_SEG columns of a row, in memory order; a thread requests all its columns before it
// uses the first.
__device__ __forceinline__ void ix_lp_widen16(const uint4 u, float (&v)[8]) { ix_unpack8(u, v); }
__device__ __forceinline__ void ix_lp_widen16(const uint4 u, float (&v)[4]) {
  v[0] = __uint_as_float(u.x); v[1] = __uint_as_float(u.y); v[2] = __uint_as_float(u.z); v[3] = __uint_as_float(u.w);
}
__device__ __forceinline__ uint4 ix_lp_pack16(const float (&v)[8]) {
  return make_uint4(ix_pack_bf2(v[0], v[1]), ix_pack_bf2(v[2], v[3]), ix_pack_bf2(v[4], v[5]), ix_pack_bf2(v[6], v[7]));
}
__device__ __forceinline__ uint4 ix_lp_pack16(const float (&v)[4]) {
  return make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3]));
}
__device__ __forceinline__ void ix_lp_store1(bf16_t* p, float v) { *p = ix_f2bf(v); }
__device__ __forceinline__ void ix_lp_store1(float* p, float v) { *p = v; }

// ONCE: the caches are too small for the logits and the gradient; both go past them.
template <typename T, bool ONCE>
__global__ __launch_bounds__(256) void k_lp_backward(const T* __restrict__ x, long row_stride, int V, int P,
                                                     const int64_t* __restrict__ target,
                                                     const float* __restrict__ upstream, const float* __restrict__ lse,
                                                     T* __restrict__ grad, long grad_stride, int vec) {
  constexpr int W = 16 / sizeof(T);  // columns of one 16-byte access; a wave's access is 1 KiB of the row
  constexpr int GROUPS = IX_LP_SEG / (256 * W);
  const long row = blockIdx.x / P;  // segments fastest
  const int lo = (int)(blockIdx.x % P) * IX_LP_SEG;
  const int hi = min(V, lo + IX_LP_SEG);
  const T* xr = x + row * row_stride;
  T* gr = grad + row * grad_stride;
  if (vec) {  // V is a multiple of 8: a group is whole or absent (an absent one reads the segment's first columns)
    uint4 raw[GROUPS];
#pragma unroll
    for (int c = 0; c < GROUPS; ++c) {
      const int off = lo + (c * 256 + (int)threadIdx.x) * W;
      const uint4* p = reinterpret_cast<const uint4*>(xr + (off < hi ? off : lo));
      raw[c] = ONCE ? ix_load16_once(p) : *p;
    }
    __builtin_amdgcn_sched_barrier(0);
    const int64_t t64 = target[row];
    const bool valid = t64 >= 0 && t64 < (int64_t)V;
    const int t = valid ? (int)t64 : -1;
    const float u = valid ? upstream[row] : 0.0f, ls = lse[row];
#pragma unroll
    for (int c = 0; c < GROUPS; ++c) {
      const int off = lo + (c * 256 + (int)threadIdx.x) * W;
      float v[W];
      ix_lp_widen16(raw[c], v);
#pragma unroll
      for (int i = 0; i < W; ++i) {
        v[i] = ix_exp(v[i] - ls) * -u;
        if (off + i == t) v[i] = v[i] + u;
      }
      if (off >= hi) continue;
      uint4* d = reinterpret_cast<uint4*>(gr + off);
      if (ONCE) ix_store16_once(d, ix_lp_pack16(v));
      else *d = ix_lp_pack16(v);
    }
    return;
  }
  const int64_t t64 = target[row];
  const bool valid = t64 >= 0 && t64 < (int64_t)V;
  const int t = valid ? (int)t64 : -1;
  const float u = valid ? upstream[row] : 0.0f, ls = lse[row];
  for (int j = lo + (int)threadIdx.x; j < hi; j += 256) {
    float o[8];
    ix_load8(xr + j, 1, false, 0.0f, o);
    float v = ix_exp(o[0] - ls) * -u;
    if (j == t) v = v + u;
    ix_lp_store1(gr + j, v);
  }
}

// rowmax[row] = max over P parts (exact; any order). One wave per row, or (many parts) one workgroup per row with all its
// loads in flight: a wave walks 2376 parts one dependent load after the other (513 rows of 2376 parts 19.7 -> 5.3 us). The line:
// up to 8192 rows the two are equal at 500 to 1000 parts; us wave / workgroup at 16384 rows 512 parts 6.9 / 9.0, 594 9.2 / 9.4, 640
// 9.5 / 9.5, 768 10.9 / 9.6, 1187 15.7 / 12.4.
#define IX_LP_MANY_PARTS 640
__global__ __launch_bounds__(256) void k_lp_reduce_parts(const float* __restrict__ parts, long parts_ld, int P,
                                                         long rows, float* __restrict__ rowmax) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float m = ix_row_max_from_parts(parts + row * parts_ld, P, threadIdx.x & 63);
  if ((threadIdx.x & 63) == 0) rowmax[row] = m;
}

__global__ __launch_bounds__(256) void k_lp_reduce_many_parts(const float* __restrict__ parts, long parts_ld, int P,
                                                              float* __restrict__ rowmax) {
  __shared__ float s_w[4];
  const long row = blockIdx.x;
  const float* pr = parts + row * parts_ld;
  float m = IX_NEG_INF;
  for (int i0 = threadIdx.x; i0 < P; i0 += 256 * 8) {
    float v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = pr[min(i0 + c * 256, P - 1)];
#pragma unroll
    for (int c = 0; c < 8; ++c) m = fmaxf(m, v[c]);
  }
  m = ix_lane_max<64>(m);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) rowmax[row] = fmaxf(fmaxf(s_w[0], s_w[1]), fmaxf(s_w[2], s_w[3]));
}

extern "C" int ix_rowmax_reduce(const float* parts, long parts_ld, long P, long rows, float* rowmax, void* stream) {
  if (!parts || !rowmax || rows < 0 || P <= 0 || parts_ld < P || P > 0x7fffffffL) return IX_ERR_ARG;
  if (rows == 0) return IX_OK;
  if (P >= IX_LP_MANY_PARTS && P <= 0x40000000L && rows <= 0x7fffffffL) {  // the walk's index runs up to 2047 past P
    hipLaunchKernelGGL(k_lp_reduce_many_parts, dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream, parts, parts_ld, (int)P,
                       rowmax);
    return ix_launch_status();
  }
  const long grid = (rows + 3) / 4;
  if (grid > 0x7fffffffL) return IX_DECLINED;
  hipLaunchKernelGGL(k_lp_reduce_parts, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, parts, parts_ld,
                     (int)P, rows, rowmax);
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
static int ix_lp_check(const void* logits, int dtype, long rows, long V, long row_stride, int G) {
  if (!logits || rows < 0 || V <= 0 || row_stride < V) return IX_ERR_ARG;
  if (dtype != IX_DT_F32 && dtype != IX_DT_BF16) return IX_DECLINED;
  if (G < 1 || G > IX_LP_MAX_G || (G & (G - 1)) != 0) return IX_DECLINED;
  if (V % G != 0) return IX_DECLINED;  // unequal leaves change the contract (rowinv.py:376-377)
  if (V > 0x7fffffffL || rows > 0x7fffffffL) return IX_DECLINED;
  const long L = V / G;
  const long NB = (L + IX_LP_BLOCK - 1) / IX_LP_BLOCK;
  if (G * NB > IX_LP_MAX_UNITS) return IX_DECLINED;
  return IX_OK;
}

extern "C" size_t ix_logprob_workspace_bytes(long rows, long V, int G) {
  if (rows <= 0 || V <= 0 || G < 1 || V % G != 0) return 0;
  const long L = V / G;
  const long NB = (L + IX_LP_BLOCK - 1) / IX_LP_BLOCK;
  const long P = (V + IX_LP_SEG - 1) / IX_LP_SEG;
  return (size_t)rows * (size_t)(P + G * NB + 2) * sizeof(float);
}

// Whether whole rows go to k_lp_row_held: us twice read (k_lp_row) / kept.
//   * 65536 columns: 1000 rows fp32 78 / 50, bf16 42 / 36; of 32000, one block a wave, 36 / 42 and 20 / 22.
//   * A group past its block's end is a load like the others. fp32: blocks half full pay (1000 rows of 131072 in 64 leaves 157 / 133,
//     257 of 65536 in 32 34 / 31), quarters do not (257 of 65536 in 64 45 / 49).
//   * fp32 gains at every row count, also just past a whole turn of the CUs, and at every width (257 x 151936 65 / 53, 1025 x 151936
//     184 / 141, 257 x 2097152 924 / 892).
//   * bf16, all blocks in registers (40): 256 x 73728 14.2 / 13.4, 257 18.5 / 18.8, 300 20.7 / 20.1; 257 x 151936 39.9 / 36.2. Below
//     73728 columns a second turn of a few rows is worse (257 x 65536 16.0 / 16.8, 300 17.6 / 17.7; 256 11.9 / 11.9, 384 19.8 / 18.9).
//   * bf16, some blocks read twice after all: 192 x 196608 29.1 / 29.1, 257 x 262144 63.8 / 64.5, 513 x 524288 204 / 207, 1025 x
//     1048576 747 / 770; but 384 x 180224 51.9 / 48.3, 384 x 393216 108 / 106, 1537 x 393216 394 / 348, 600 x 524288 227 / 215. Blocks
//     three quarters full are then not enough (513 x 196608 in 32 leaves 84 / 87).
extern "C" int ix_logprob_keeps_rows(int dtype, long rows, long V, int G) {
  if (G < 1 || V < 65536 || V % G != 0) return 0;
  const long units = G * ((V / G + IX_LP_BLOCK - 1) / IX_LP_BLOCK), columns = units * IX_LP_BLOCK;
  if (units > IX_LP_HELD_UNITS || rows < IX_LP_SPLIT_BELOW) return 0;
  if (dtype != IX_DT_BF16) return 2 * V >= columns;
  if (units <= 40) return V >= 73728 || rows <= 256 || rows >= 384;
  return units <= (rows >= 576 ? 128 : 96) && rows >= 384 && 8 * V >= 7 * columns;
}

template <typename T>
static int ix_lp_launch(const T* x, long rows, long V, long row_stride, int G, const int64_t* target,
                        float* out_lp, float* out_lse, float* out_full, long full_stride, float* ws,
                        size_t ws_bytes, int force_shape, const float* row_max_in, hipStream_t st) {
  if (rows == 0) return IX_OK;
  const long L = V / G;
  const int vec = (ix_aligned(x, 8 * sizeof(T)) && (row_stride % 8 == 0) && (L % 8 == 0)) ? 1 : 0;
  // a caller-supplied row max (exact, e.g. from the producing GEMM's epilogue) removes the max
  // pass: the row is then read from HBM once, by the block sums
  const bool split = row_max_in || force_shape == 2 || (force_shape == 0 && rows < IX_LP_SPLIT_BELOW);
  const bool can_keep = vec && !out_full && !row_max_in && G * ((L + IX_LP_BLOCK - 1) / IX_LP_BLOCK) <= IX_LP_HELD_UNITS;
  if (force_shape == 3 && !can_keep) return IX_DECLINED;
  if (force_shape == 3 ||
      (force_shape == 0 && can_keep && ix_logprob_keeps_rows(sizeof(T) == 2 ? IX_DT_BF16 : IX_DT_F32, rows, V, G))) {
    constexpr int HU = sizeof(T) == 2 ? 5 : 2, LU = sizeof(T) == 2 ? 0 : 1;
    hipLaunchKernelGGL((k_lp_row_held<T, HU, LU>), dim3((unsigned)(rows < 256 ? rows : 256)), dim3(512),
                       (size_t)LU * 8 * IX_LP_BLOCK * sizeof(T), st, x, row_stride, rows, (int)V, G, target, out_lp, out_lse);
    return ix_launch_status();
  }
  if (!split) {
    hipLaunchKernelGGL((k_lp_row<T>), dim3((unsigned)rows), dim3(512), 0, st, x, row_stride, (int)V, G, target,
                       out_lp, out_lse, out_full, full_stride, vec);
    return ix_launch_status();
  }
  if (rows * (long)((V + IX_LP_SEG - 1) / IX_LP_SEG) > 0x7fffffffL || rows * (long)(G * ((L + IX_LP_BLOCK - 1) / IX_LP_BLOCK)) > 0x7fffffffL)
    return IX_DECLINED;
  if (!ws || ws_bytes < ix_logprob_workspace_bytes(rows, V, G)) return IX_ERR_ARG;
  const int NB = (int)((L + IX_LP_BLOCK - 1) / IX_LP_BLOCK);
  const int PW = (int)((V + IX_LP_SEG - 1) / IX_LP_SEG);  // workspace layout always reserves PW parts
  const int U = G * NB;
  float* ws_pmax = ws;
  float* bsum = ws_pmax + rows * PW;
  const int P = row_max_in ? 1 : PW;
  const float* pmax = row_max_in ? row_max_in : ws_pmax;
  if (!row_max_in)
    hipLaunchKernelGGL((k_lp_partmax<T>), dim3((unsigned)(rows * P)), dim3(256), 0, st, x, row_stride, (int)V, P,
                       ws_pmax, vec);
  const int ny = (U + 3) / 4;
  const unsigned total = (unsigned)(rows * ny);
  hipLaunchKernelGGL((k_lp_blocksums<T>), dim3(ix_xcd_run_grid(total)), dim3(256), 0, st, x, row_stride, (int)V, G,
                     P, pmax, bsum, vec, ny, total);
  float* fin = out_full && ix_lp_joins_in_front(rows, NB) ? bsum + rows * U : nullptr;
  if (!out_full || fin)
    hipLaunchKernelGGL((k_lp_finalize<T>), dim3((unsigned)rows), dim3(64), 0, st, x, row_stride, (int)V, G, P, pmax,
                       bsum, fin, target, out_lp, out_lse);
  if (!out_full) return ix_launch_status();
  const int vec4 = vec && full_stride % 4 == 0 && ix_aligned(out_full, 16);
  hipLaunchKernelGGL((k_lp_fullwrite<T>), dim3((unsigned)(rows * PW)), dim3(256), 0, st, x, row_stride, (int)V, G, P, pmax,
                     bsum, fin, out_full, full_stride, out_lse, vec4, PW);
  return ix_launch_status();
}

extern "C" int ix_logprob_rowinv_sampled(const void* logits, int dtype, long rows, long V, long row_stride,
                                         const int64_t* target, int G, float* out_logprob, float* out_lse,
                                         void* workspace, size_t workspace_bytes, int force_shape,
                                         const float* row_max_in, void* stream) {
  int rc = ix_lp_check(logits, dtype, rows, V, row_stride, G);
  if (rc != IX_OK) return rc;
  if (!target || !out_logprob) return IX_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == IX_DT_BF16)
    return ix_lp_launch((const bf16_t*)logits, rows, V, row_stride, G, target, out_logprob, out_lse, nullptr, 0,
                        (float*)workspace, workspace_bytes, force_shape, row_max_in, st);
  return ix_lp_launch((const float*)logits, rows, V, row_stride, G, target, out_logprob, out_lse, nullptr, 0,
                      (float*)workspace, workspace_bytes, force_shape, row_max_in, st);
}

extern "C" int ix_logprob_rowinv_full(const void* logits, int dtype, long rows, long V, long row_stride, int G,
                                      float* out_full, long out_stride, float* out_lse, void* workspace,
                                      size_t workspace_bytes, int force_shape, const float* row_max_in,
                                      void* stream) {
  int rc = ix_lp_check(logits, dtype, rows, V, row_stride, G);
  if (rc != IX_OK) return rc;
  if (!out_full || out_stride < V) return IX_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == IX_DT_BF16)
    return ix_lp_launch((const bf16_t*)logits, rows, V, row_stride, G, nullptr, nullptr, out_lse, out_full,
                        out_stride, (float*)workspace, workspace_bytes, force_shape, row_max_in, st);
  return ix_lp_launch((const float*)logits, rows, V, row_stride, G, nullptr, nullptr, out_lse, out_full,
                      out_stride, (float*)workspace, workspace_bytes, force_shape, row_max_in, st);
}

extern "C" int ix_logprob_rowinv_backward(const void* logits, int dtype, long rows, long V, long row_stride,
                                          const int64_t* target, const float* upstream, const float* lse, void* grad,
                                          long grad_stride, void* stream) {
  if (!logits || !target || !upstream || !lse || !grad || rows < 0 || V <= 0 || row_stride < V || grad_stride < V)
    return IX_ERR_ARG;
  if (dtype != IX_DT_F32 && dtype != IX_DT_BF16) return IX_DECLINED;
  if (rows == 0) return IX_OK;
  const long P = (V + IX_LP_SEG - 1) / IX_LP_SEG;
  if (V > 0x7fff0000L || rows * P > 0x7fffffffL) return IX_DECLINED;
  const int vec = (V % 8 == 0) && (row_stride % 8 == 0) && (grad_stride % 8 == 0) && ix_aligned(logits, 16) && ix_aligned(grad, 16);
  // Logits of 256 MiB and more (the memory-side cache): a default store leaves dirty lines that the next kernel's reads
  // have to wait for, and a default load only displaces lines. Forward + backward, us, default / past the caches: fp32
  // 1000 rows of 151936 413 / 367, 2900 1165 / 1086, bf16 1000 217 / 200, 2900 602 / 572; below the line the logits are
  // still there for the next pass (fp32 300 rows 122 / 124, 100 rows 48 / 51).
  const bool once = rows * V * (long)(dtype == IX_DT_BF16 ? sizeof(bf16_t) : sizeof(float)) >= (256L << 20);
  hipStream_t st = (hipStream_t)stream;
#define IX_LP_BACK(T, ONCE)                                                                                         \
  hipLaunchKernelGGL((k_lp_backward<T, ONCE>), dim3((unsigned)(rows * P)), dim3(256), 0, st, (const T*)logits, row_stride, \
                     (int)V, (int)P, target, upstream, lse, (T*)grad, grad_stride, vec)
  if (dtype == IX_DT_BF16) {
    if (once) IX_LP_BACK(bf16_t, true);
    else IX_LP_BACK(bf16_t, false);
  } else {
    if (once) IX_LP_BACK(float, true);
    else IX_LP_BACK(float, false);
  }
#undef IX_LP_BACK
  return ix_launch_status();
}
