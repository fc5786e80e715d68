// Mixture-of-experts FFN: router top-k, expert-major permutation and block map, grouped
// fc1 + SwiGLU + prob epilogue, grouped fc2, fixed-order combine.
//
// Per-token function (skyrl/backends/skyrl_train/isoexec/ops/moe/moe_router_o2_kernel.py:87-174,369-386,
// moe_batched_experts.py:496-503, moe_batch_invariant.py:276-320, moe_combine_kernel.py:36-76):
//   router : k winners by (score desc, expert index asc); NaN scores count as -inf
//            mode 0: p = softmax over the k winning logits            (top-k then softmax)
//            mode 1: softmax over all E, top-k on the probabilities, renormalise by their sum
//            both sums over the k winners: adjacent-pairwise tree in rank order
//   expert : inter = bf16(x W1^T); gate/up halves; s = bf16(gate / (1 + exp(-gate)));
//            h = bf16(s * up); a = bf16(h * prob); y = bf16(a W2^T)
//   combine: the token's k rows added in ascending expert order; bf16 adds (a round per add)
//            or one fp32 sum and a single round.
// Nothing a token sees depends on the other tokens of the batch: the permutation and the block
// map are integer-only and only decide which workgroup computes a row; the GEMM core's K order
// is fixed (ix_gemm_core.h).
#include "ix_gemm_core.h"
#include "ix_moe_bands.h"
#include "../../include/isoexec_hip.h"

#define IX_MOE_KMAX 16
#define IX_MOE_EC 8  // experts per lane: E <= 512
#define IX_MOE_TILE_T 256
#define IX_MOE_EMAX 512

// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ bool ix_beats(float av, int ai, float bv, int bi, int sentinel) {
  // does candidate a beat candidate b?  sentinel index = "no candidate"
  if (ai == sentinel) return false;
  if (bi == sentinel) return true;
  return (av > bv) || (av == bv && ai < bi);
}

// One step of the wave-wide "best candidate" exchange at lane distance S (selection by ix_beats is associative
// and commutative, so the exchange network does not matter; distances below 16 use the row-local lane controls).
template <int S>
__device__ __forceinline__ void ix_best_step(float& bv, int& bi, int sentinel) {
  const float ov = ix_xor_lane<S>(bv);
  const int oi = __float_as_int(ix_xor_lane<S>(__int_as_float(bi)));
  if (ix_beats(ov, oi, bv, bi, sentinel)) { bv = ov; bi = oi; }
}

// Minimum over the 16 lanes of a row.
__device__ __forceinline__ int ix_row_min(int v) {
  v = min(v, __float_as_int(ix_partner<1>(__int_as_float(v))));
  v = min(v, __float_as_int(ix_partner<2>(__int_as_float(v))));
  v = min(v, __float_as_int(ix_partner<4>(__int_as_float(v))));
  return min(v, __float_as_int(ix_partner<8>(__int_as_float(v))));
}

// Inclusive sum over the lanes of a wave: within rows by shifts, then each row's total into the rows above it.
__device__ __forceinline__ int ix_wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

__device__ __forceinline__ float ix_tree_k(float (&t)[IX_MOE_KMAX], int k) {
#pragma unroll
  for (int s = 1; s < IX_MOE_KMAX; s <<= 1) {
    if (s < k) {
#pragma unroll
      for (int i = 0; i < IX_MOE_KMAX; i += 2 * s)
        if (i + s < k) t[i] = t[i] + t[i + s];
    }
  }
  return t[0];
}

// EC = experts held per lane (E <= 64 EC): the instantiation only sets how many slots a lane carries.
template <int EC>
__global__ __launch_bounds__(256) void k_moe_router(const float* __restrict__ logits, long ld, int T, int E, int k,
                                                    int mode, float scaling, int* __restrict__ topk_idx,
                                                    float* __restrict__ topk_prob, float* __restrict__ dense_probs,
                                                    uint8_t* __restrict__ dense_map) {
  const int lane = threadIdx.x & 63;
  const long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  float s[EC];
  bool live[EC];
#pragma unroll
  for (int c = 0; c < EC; ++c) {
    const int e = lane + 64 * c;
    live[c] = e < E;
    float v = live[c] ? logits[t * ld + e] : IX_NEG_INF;
    if (v != v) v = IX_NEG_INF;
    s[c] = v;
  }
  if (mode == 1) {
    float m = IX_NEG_INF;
#pragma unroll
    for (int c = 0; c < EC; ++c) m = fmaxf(m, s[c]);
    m = ix_lane_max<64>(m);
    float z = 0.0f;
#pragma unroll
    for (int c = 0; c < EC; ++c) {
      s[c] = live[c] ? ix_exp(s[c] - m) : 0.0f;
      z = z + s[c];
    }
    z = ix_lane_tree<64>(z);
#pragma unroll
    for (int c = 0; c < EC; ++c) s[c] = s[c] / z;
  }
  float vals[IX_MOE_KMAX];
  int idxs[IX_MOE_KMAX];
#pragma unroll
  for (int j = 0; j < IX_MOE_KMAX; ++j) {
    vals[j] = 0.0f;
    idxs[j] = 0;
    if (j < k) {
      float bv = 0.0f;
      int bi = E;
#pragma unroll
      for (int c = 0; c < EC; ++c) {
        const int e = lane + 64 * c;
        if (live[c] && ix_beats(s[c], e, bv, bi, E)) { bv = s[c]; bi = e; }
      }
      ix_best_step<1>(bv, bi, E);
      ix_best_step<2>(bv, bi, E);
      ix_best_step<4>(bv, bi, E);
      ix_best_step<8>(bv, bi, E);
      ix_best_step<16>(bv, bi, E);
      ix_best_step<32>(bv, bi, E);
      bi = min(bi, E - 1);
      vals[j] = bv;
      idxs[j] = bi;
#pragma unroll
      for (int c = 0; c < EC; ++c)
        if (lane + 64 * c == bi) live[c] = false;
    }
  }
  float p[IX_MOE_KMAX], tmp[IX_MOE_KMAX];
  if (mode == 0) {
    const float m = vals[0];
#pragma unroll
    for (int j = 0; j < IX_MOE_KMAX; ++j) { p[j] = (j < k) ? ix_exp(vals[j] - m) : 0.0f; tmp[j] = p[j]; }
  } else {
#pragma unroll
    for (int j = 0; j < IX_MOE_KMAX; ++j) { p[j] = (j < k) ? vals[j] : 0.0f; tmp[j] = p[j]; }
  }
  const float den = ix_tree_k(tmp, k);
#pragma unroll
  for (int j = 0; j < IX_MOE_KMAX; ++j) {
    p[j] = p[j] / den;
    if (scaling != 0.0f) p[j] = p[j] * scaling;
  }
#pragma unroll
  for (int j = 0; j < IX_MOE_KMAX; ++j) {
    if (j < k && lane == j) {
      topk_idx[t * k + j] = idxs[j];
      topk_prob[t * k + j] = p[j];
    }
  }
  if (dense_probs || dense_map) {
#pragma unroll
    for (int c = 0; c < EC; ++c) {
      const int e = lane + 64 * c;
      if (e < E) {
        float dp = 0.0f;
        uint8_t dm = 0;
#pragma unroll
        for (int j = 0; j < IX_MOE_KMAX; ++j)
          if (j < k && idxs[j] == e) { dp = p[j]; dm = 1; }
        if (dense_probs) dense_probs[t * E + e] = dp;
        if (dense_map) dense_map[t * E + e] = dm;
      }
    }
  }
}

// E <= 128: a token takes 16 lanes (a row of the wave, so every exchange is a row-local lane control) and a wave
// routes 4 tokens. Lane i of the row holds experts 4i .. 4i+3 and 64+4i .. 64+4i+3. Same function as k_moe_router
// bit for bit: the winner under ix_beats does not depend on the exchange network, and the softmax denominator is
// built as there -- s[v] + s[v + 64] per v = e mod 64, then the adjacent-pairwise tree over v (two levels inside the
// lane, four across the row).
// Token t by the 16 lanes of one row of a wave (li = lane within the row). Called with whole rows only (every lane of
// a row has the same t), so the lane controls below stay inside live lanes.
__device__ __forceinline__ void ix_moe_route_row16(const float* __restrict__ logits, long ld, long t, int li, int E,
                                                   int k, int mode, float scaling, int* __restrict__ topk_idx,
                                                   float* __restrict__ topk_prob, float* __restrict__ dense_probs,
                                                   uint8_t* __restrict__ dense_map, int* __restrict__ lds_idx,
                                                   float* __restrict__ lds_prob) {
  float s[8];
  int eid[8];
  bool live[8];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int e0 = 64 * h + 4 * li;
    float4 v4 = make_float4(IX_NEG_INF, IX_NEG_INF, IX_NEG_INF, IX_NEG_INF);
    if (e0 + 4 <= E && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0) {
      v4 = *reinterpret_cast<const float4*>(logits + t * ld + e0);
    } else {
      if (e0 + 0 < E) v4.x = logits[t * ld + e0 + 0];
      if (e0 + 1 < E) v4.y = logits[t * ld + e0 + 1];
      if (e0 + 2 < E) v4.z = logits[t * ld + e0 + 2];
      if (e0 + 3 < E) v4.w = logits[t * ld + e0 + 3];
    }
    const float q[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int e = e0 + c;
      eid[4 * h + c] = e;
      live[4 * h + c] = e < E;
      float v = live[4 * h + c] ? q[c] : IX_NEG_INF;
      if (v != v) v = IX_NEG_INF;
      s[4 * h + c] = v;
    }
  }
  if (mode == 1) {
    float m = IX_NEG_INF;
#pragma unroll
    for (int c = 0; c < 8; ++c) m = fmaxf(m, s[c]);
    m = ix_lane_max<16>(m);
    float zl[4];
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = live[c] ? ix_exp(s[c] - m) : 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) zl[c] = s[c] + s[4 + c];
    float z = (zl[0] + zl[1]) + (zl[2] + zl[3]);
    z = ix_lane_tree<16>(z);
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = s[c] / z;
  }
  // k rounds of "the largest value left, the lowest expert among equals" (ix_beats). A round is a maximum over the row and a
  // minimum over the experts that reach it, both of which ride the vector ALU's lane controls as one instruction a step
  // (value and index exchanged as a pair and compared cost twice the instructions; at 64 tokens four waves share a SIMD and
  // issue is what a round costs). A taken or missing expert is a NaN: the maximum passes it over and nothing equals it.
  // Scores that are NaN (an infinite logit under mode 1: then the whole row is) rank with -inf.
  const float none = __uint_as_float(0x7fc00000u);
  float sel[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) sel[c] = live[c] ? (s[c] != s[c] ? IX_NEG_INF : s[c]) : none;
  float top = 0.0f, mine = 0.0f;  // round 0's value; lane j of the row keeps round j's
  int mine_e = 0;
#pragma unroll
  for (int j = 0; j < IX_MOE_KMAX; ++j) {
    if (j < k) {
      const float m = ix_lane_max<16>(fmaxf(fmaxf(fmaxf(sel[0], sel[1]), fmaxf(sel[2], sel[3])),
                                            fmaxf(fmaxf(sel[4], sel[5]), fmaxf(sel[6], sel[7]))));
      int bi = IX_MOE_EMAX;  // no expert of this lane
#pragma unroll
      for (int c = 7; c >= 0; --c) bi = sel[c] == m ? eid[c] : bi;  // eid[] ascends
      bi = ix_row_min(bi);
      if (j == 0) top = m;
      if (li == j) { mine = m; mine_e = bi; }
#pragma unroll
      for (int c = 0; c < 8; ++c) sel[c] = eid[c] == bi ? none : sel[c];
    }
  }
  // lane j < k holds winner j; the tree over k lanes goes on over zeros, which change no bit of a sum of non-negatives
  float p = li < k ? (mode == 0 ? ix_exp(mine - top) : mine) : 0.0f;
  p = p / ix_lane_tree<16>(p);
  if (scaling != 0.0f) p = p * scaling;
  if (li < k) {
    topk_idx[t * k + li] = mine_e;
    topk_prob[t * k + li] = p;
    if (lds_idx) {  // a kernel that goes on to permute keeps the winners in LDS as well
      lds_idx[t * k + li] = mine_e;
      lds_prob[t * k + li] = p;
    }
  }
  if (dense_probs || dense_map) {
    float dp[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    uint8_t dm[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int j = 0; j < k; ++j) {
      const int ej = __shfl(mine_e, j, 16);
      const float pj = __shfl(p, j, 16);
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (ej == eid[c]) { dp[c] = pj; dm[c] = 1; }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int e = eid[c];
      if (e < E) {
        if (dense_probs) dense_probs[t * E + e] = dp[c];
        if (dense_map) dense_map[t * E + e] = dm[c];
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_moe_router_row16(const float* __restrict__ logits, long ld, int T, int E,
                                                          int k, int mode, float scaling, int* __restrict__ topk_idx,
                                                          float* __restrict__ topk_prob,
                                                          float* __restrict__ dense_probs,
                                                          uint8_t* __restrict__ dense_map) {
  const long t = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (t >= T) return;  // whole rows leave together
  ix_moe_route_row16(logits, ld, t, threadIdx.x & 15, E, k, mode, scaling, topk_idx, topk_prob, dense_probs, dense_map,
                     nullptr, nullptr);
}

extern "C" int ix_moe_router_topk(const float* logits, long ld, long T, long E, long k, int mode, float scaling,
                                  int* topk_idx, float* topk_prob, float* dense_probs, uint8_t* dense_map,
                                  void* stream) {
  if (!logits || !topk_idx || !topk_prob || T < 0 || E <= 0 || k <= 0 || ld < E) return IX_ERR_ARG;
  if (k > E || k > IX_MOE_KMAX || (k & (k - 1)) != 0) return IX_DECLINED;  // pow2 k: padding would re-associate
  if (E > 64 * IX_MOE_EC) return IX_DECLINED;
  if (mode != 0 && mode != 1) return IX_ERR_ARG;
  if (T == 0) return IX_OK;
  const long grid = (T + 3) / 4;
  if (grid > 0x7fffffffL) return IX_DECLINED;
#define IX_ROUTER(EC_)                                                                                            \
  hipLaunchKernelGGL(k_moe_router<EC_>, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, logits, ld,      \
                     (int)T, (int)E, (int)k, mode, scaling, topk_idx, topk_prob, dense_probs, dense_map)
  if (E <= 128) {
    const long grid16 = (T + 15) / 16;
    hipLaunchKernelGGL(k_moe_router_row16, dim3((unsigned)grid16), dim3(256), 0, (hipStream_t)stream, logits, ld,
                       (int)T, (int)E, (int)k, mode, scaling, topk_idx, topk_prob, dense_probs, dense_map);
  } else if (E <= 256) IX_ROUTER(4);
  else IX_ROUTER(IX_MOE_EC);
#undef IX_ROUTER
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// Permutation (integer only). Token tiles of 256. Per tile and expert, a 256-bit membership mask
// is built in LDS with integer OR (order-free, so the mask is the same in any execution order);
// a row's position inside its expert's segment is then a popcount of the mask below the token,
// which makes every expert's rows token-ascending without any ordered loop or counter.
__device__ __forceinline__ void ix_moe_build_masks(const int* __restrict__ topk_idx, int t0, int nt, int E, int k,
                                                   uint32_t* s_mask /* [E][8] */, int* s_idx /* [256][k] */) {
  const int nthreads = blockDim.x;
  for (int i = threadIdx.x; i < E * 8; i += nthreads) s_mask[i] = 0u;
  for (int i = threadIdx.x; i < nt * k; i += nthreads) s_idx[i] = topk_idx[(long)t0 * k + i];
  __syncthreads();
  for (int i = threadIdx.x; i < nt * k; i += nthreads) {
    const int t = i / k;
    atomicOr(&s_mask[s_idx[i] * 8 + (t >> 5)], 1u << (t & 31));
  }
  __syncthreads();
}

__global__ __launch_bounds__(256) void k_moe_tile_counts(const int* __restrict__ topk_idx, int T, int E, int k,
                                                         int* __restrict__ tile_counts) {
  __shared__ int s_idx[IX_MOE_TILE_T * IX_MOE_KMAX];
  __shared__ uint32_t s_mask[IX_MOE_EMAX * 8];
  const int tile = blockIdx.x;
  const int t0 = tile * IX_MOE_TILE_T;
  const int nt = min(IX_MOE_TILE_T, T - t0);
  ix_moe_build_masks(topk_idx, t0, nt, E, k, s_mask, s_idx);
  for (int e = threadIdx.x; e < E; e += 256) {
    int c = 0;
#pragma unroll
    for (int w = 0; w < 8; ++w) c += __popc(s_mask[e * 8 + w]);
    tile_counts[(long)tile * E + e] = c;
  }
}

// Per expert, the running sum of its counts over the token tiles (tile_base[t][e] = rows of expert e in tiles before t)
// and its total. One wave per expert: a lane owns a run of consecutive tiles, sums it, the lanes' sums are scanned across
// the wave, then the lane walks its run again writing the bases. Integer only.
__global__ __launch_bounds__(256) void k_moe_tile_prefix(const int* __restrict__ tile_counts, int ntiles, int E,
                                                         int* __restrict__ tile_base, int* __restrict__ counts) {
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= E) return;  // whole waves leave together
  const int lane = threadIdx.x & 63;
  const int per = (ntiles + 63) >> 6;
  const int t_lo = min(lane * per, ntiles), t_hi = min(t_lo + per, ntiles);
  int mine = 0;
  for (int t = t_lo; t < t_hi; ++t) mine += tile_counts[(long)t * E + e];
  int incl = mine;  // inclusive scan over the lanes
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(incl, d, 64);
    if (lane >= d) incl += up;
  }
  int run = incl - mine;
  for (int t = t_lo; t < t_hi; ++t) {
    const int c = tile_counts[(long)t * E + e];
    tile_base[(long)t * E + e] = run;
    run += c;
  }
  if (lane == 63) counts[e] = incl;
}

// meta layout: [0] = number of m-tiles, then tile_expert[max_tiles], tile_row0[max_tiles], tile_nrows[max_tiles]. The row
// tiles of expert e: c rows from row0 on, its first tile number nt.
__device__ __forceinline__ void ix_moe_write_tiles(int e, int c, int row0, int nt, int BM, int max_tiles, int* meta) {
  int* tile_expert = meta + 1;
  int* tile_row0 = tile_expert + max_tiles;
  int* tile_nrows = tile_row0 + max_tiles;
  for (int r0 = 0; r0 < c && nt < max_tiles; r0 += BM, ++nt) {
    tile_expert[nt] = e;
    tile_row0[nt] = row0 + r0;
    tile_nrows[nt] = min(BM, c - r0);
  }
}

// A second map of 256-row tiles beside one of 160 or 192, of which the counts decide which is used (the other gets no
// tiles). The kernels of both heights are launched; those of the empty map find no tile and exit.
struct IxMoeTall {
  int* meta;               // null: the map has one height
  int max_tiles;
  float us_low;            // what the first map's tiles cost
  int nb1, kt1, nb2, kt2;  // column tiles and k-tiles of the two products
};

// What both products cost with `tiles` row tiles at `us` per k-tile: turns of the chip's 256 workgroups, where a last turn that
// is not full costs two thirds of one and the rest by its share. `us` is a fit to 737 launches (seventeen layers, three
// routings, 24 to 400 rows per expert) whose times it gives with a deviation of 6 %.
#define IX_MOE_US_160 1.27f
#define IX_MOE_US_192 1.41f
#define IX_MOE_US_256 1.64f
__device__ __forceinline__ float ix_moe_tiles_cost(const IxMoeTall& h, int tiles, float us) {
  auto turns = [](float t) {
    const float full = floorf(t);
    return t > full ? full + 0.68f + 0.32f * (t - full) : full;
  };
  return us * (turns((float)tiles * (float)h.nb1 / 256.0f) * (float)h.kt1 +
               turns((float)tiles * (float)h.nb2 / 256.0f) * (float)h.kt2);
}

// Exclusive scans over the experts by one wave (rows and row tiles; s_cnt is zero past the last expert): a lane owns EMAX / 64
// consecutive ones. Returns the rows of a tile: BM, or 256 where the counts decide for the tall map. `write`: also the total to
// offsets[E] (if there are offsets) and the number of tiles to the maps.
__device__ __forceinline__ int ix_moe_scan_experts(const int* s_cnt, int E, int BM, int max_tiles, const IxMoeTall& tall,
                                                   int* s_off, int* s_toff, bool write, int* offsets, int* meta) {
  constexpr int PER = IX_MOE_EMAX / 64;
  const int lane = threadIdx.x;
  auto count = [&](int rows_per_tile, int& rows, int& tiles) {  // this lane's experts, then all up to them
    rows = tiles = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = s_cnt[lane * PER + i];
      rows += c;
      tiles += (c + rows_per_tile - 1) / rows_per_tile;
    }
    const int own_rows = rows, own_tiles = tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int a = __shfl_up(rows, d, 64), b = __shfl_up(tiles, d, 64);
      if (lane >= d) { rows += a; tiles += b; }
    }
    return make_int2(rows - own_rows, tiles - own_tiles);
  };
  int rows, tiles;
  int2 before = count(BM, rows, tiles);
  int total = __shfl(tiles, 63, 64);
  bool is_tall = false;
  if (tall.meta) {
    int tall_tiles;
    const int2 b = count(256, rows, tall_tiles);
    const int tall_total = __shfl(tall_tiles, 63, 64);
    is_tall = ix_moe_tiles_cost(tall, tall_total, IX_MOE_US_256) <= ix_moe_tiles_cost(tall, total, tall.us_low);
    if (write && lane == 0) {
      meta[0] = is_tall ? 0 : min(total, max_tiles);
      tall.meta[0] = is_tall ? min(tall_total, tall.max_tiles) : 0;
    }
    if (is_tall) { before = b; BM = 256; }
  } else if (write && lane == 0) {
    meta[0] = min(total, max_tiles);
  }
  if (write && offsets && lane == 63) offsets[E] = rows;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = s_cnt[lane * PER + i];
    s_off[lane * PER + i] = before.x;
    s_toff[lane * PER + i] = before.y;
    before.x += c;
    before.y += (c + BM - 1) / BM;
  }
  return BM;
}

// The row tiles of every expert and its offset, from those scans, by the whole workgroup.
__device__ __forceinline__ void ix_moe_write_map(const int* s_cnt, const int* s_off, const int* s_toff, int E, int rows_per_tile,
                                                 int BM, int max_tiles, const IxMoeTall& tall, int* offsets, int* meta) {
  const bool is_tall = rows_per_tile != BM;
  for (int e = threadIdx.x; e < E; e += (int)blockDim.x) {
    if (offsets) offsets[e] = s_off[e];
    ix_moe_write_tiles(e, s_cnt[e], s_off[e], s_toff[e], rows_per_tile, is_tall ? tall.max_tiles : max_tiles,
                       is_tall ? tall.meta : meta);
  }
}

// One workgroup, after k_moe_tile_prefix has left every expert's row count in `counts`.
__global__ __launch_bounds__(256) void k_moe_offsets(int E, int BM, int max_tiles, IxMoeTall tall,
                                                     const int* __restrict__ counts, int* __restrict__ offsets,
                                                     int* __restrict__ meta) {
  __shared__ int s_cnt[IX_MOE_EMAX], s_off[IX_MOE_EMAX], s_toff[IX_MOE_EMAX], s_rows_per_tile;
  const int tid = threadIdx.x;
  for (int e = tid; e < IX_MOE_EMAX; e += 256) s_cnt[e] = e < E ? counts[e] : 0;
  __syncthreads();
  if (tid < 64) {
    const int r = ix_moe_scan_experts(s_cnt, E, BM, max_tiles, tall, s_off, s_toff, true, offsets, meta);
    if (tid == 0) s_rows_per_tile = r;
  }
  __syncthreads();
  ix_moe_write_map(s_cnt, s_off, s_toff, E, s_rows_per_tile, BM, max_tiles, tall, offsets, meta);
}

// 1024 threads, a (token, choice) pair at a time: bound by the latency of a pair's lookups (10 us with a token per thread
// that walks its choices one after the other). base(e): the expert's first row of this token tile.
template <typename Base>
__device__ __forceinline__ void ix_moe_scatter_tile(int t0, int nt, int k, const uint32_t* s_mask, const int* s_idx,
                                                    const float* topk_prob, const Base& base, int* sorted_token,
                                                    float* permuted_prob, int* combine_rows) {
  for (int i = threadIdx.x; i < nt * k; i += 1024) {
    const int t = i / k, e = s_idx[i];
    const long first = (long)t0 * k;
    int local = __popc(s_mask[e * 8 + (t >> 5)] & ((1u << (t & 31)) - 1u));
    for (int w = 0; w < (t >> 5); ++w) local += __popc(s_mask[e * 8 + w]);
    int rank = 0;
    for (int j2 = 0; j2 < k; ++j2) rank += (s_idx[t * k + j2] < e);
    const int pos = base(e) + local;
    sorted_token[pos] = t0 + t;
    permuted_prob[pos] = topk_prob[first + i];
    combine_rows[first + t * k + rank] = pos;
  }
}

__global__ __launch_bounds__(1024) void k_moe_scatter(const int* __restrict__ topk_idx,
                                                     const float* __restrict__ topk_prob, int T, int E, int k,
                                                     const int* __restrict__ tile_base,
                                                     const int* __restrict__ offsets, int* __restrict__ sorted_token,
                                                     float* __restrict__ permuted_prob,
                                                     int* __restrict__ combine_rows) {
  __shared__ int s_idx[IX_MOE_TILE_T * IX_MOE_KMAX];
  __shared__ uint32_t s_mask[IX_MOE_EMAX * 8];
  const int tile = blockIdx.x;
  const int t0 = tile * IX_MOE_TILE_T;
  const int nt = min(IX_MOE_TILE_T, T - t0);
  ix_moe_build_masks(topk_idx, t0, nt, E, k, s_mask, s_idx);
  ix_moe_scatter_tile(t0, nt, k, s_mask, s_idx, topk_prob,
                      [&](int e) { return offsets[e] + tile_base[(long)tile * E + e]; }, sorted_token, permuted_prob,
                      combine_rows);
}

// Scatter with the prefix over the token tiles and the expert offsets in the same launch, for up to IX_MOE_FEW_TILES token
// tiles and IX_MOE_FEW_COUNTS counts: every workgroup adds up the whole count table for itself (ntiles x E integers out of
// the L2) instead of waiting for two more launches of one dependent chain each; the first one also writes counts, offsets
// and the block map. Bound by those launches' latencies: prefix + offsets + scatter 15.8 -> 7.2 us at 512 tokens, 19.1 ->
// 10.7 at 4096 (128 experts), the gaps between them not counted. The table that every workgroup reads sets the line: of 512
// experts, top-8, 8192 tokens (16384 integers) 17.0 -> 15.5 us, 12000 (24064) 17.4 -> 17.4, 16384 (32768) 18.1 -> 19.8.
#define IX_MOE_FEW_TILES 64
#define IX_MOE_FEW_COUNTS 24576
__global__ __launch_bounds__(1024) void k_moe_offsets_scatter(const int* __restrict__ topk_idx,
                                                              const float* __restrict__ topk_prob, int T, int E, int k,
                                                              int ntiles, int BM, int max_tiles, IxMoeTall tall,
                                                              const int* __restrict__ tile_counts, int* __restrict__ counts,
                                                              int* __restrict__ offsets, int* __restrict__ meta,
                                                              int* __restrict__ sorted_token,
                                                              float* __restrict__ permuted_prob,
                                                              int* __restrict__ combine_rows) {
  __shared__ int s_idx[IX_MOE_TILE_T * IX_MOE_KMAX];
  __shared__ uint32_t s_mask[IX_MOE_EMAX * 8];
  __shared__ int s_cnt[IX_MOE_EMAX], s_before[IX_MOE_EMAX], s_off[IX_MOE_EMAX], s_toff[IX_MOE_EMAX], s_rows_per_tile;
  const int tid = threadIdx.x, tile = blockIdx.x;
  const int t0 = tile * IX_MOE_TILE_T;
  const int nt = min(IX_MOE_TILE_T, T - t0);
  for (int e = tid; e < IX_MOE_EMAX; e += 1024) s_cnt[e] = s_before[e] = 0;
  ix_moe_build_masks(topk_idx, t0, nt, E, k, s_mask, s_idx);  // ends with a barrier
  // threads e + E g (g < 1024 / E groups) sum expert e's counts over the token tiles g, g + groups, ..
  const int groups = 1024 / E, g = tid / E, e = tid - g * E;
  if (g < groups) {
    int all = 0, before = 0;
    for (int t = g; t < ntiles; t += groups) {
      const int c = tile_counts[t * E + e];
      all += c;
      before += t < tile ? c : 0;
    }
    atomicAdd(&s_cnt[e], all);  // integers: the order is free
    atomicAdd(&s_before[e], before);
  }
  __syncthreads();
  if (tid < 64) {
    const int r = ix_moe_scan_experts(s_cnt, E, BM, max_tiles, tall, s_off, s_toff, tile == 0, offsets, meta);
    if (tid == 0) s_rows_per_tile = r;
  }
  __syncthreads();
  if (tile == 0) {
    for (int x = tid; x < E; x += 1024) counts[x] = s_cnt[x];
    ix_moe_write_map(s_cnt, s_off, s_toff, E, s_rows_per_tile, BM, max_tiles, tall, offsets, meta);
  }
  ix_moe_scatter_tile(t0, nt, k, s_mask, s_idx, topk_prob, [&](int x) { return s_off[x] + s_before[x]; }, sorted_token,
                      permuted_prob, combine_rows);
}

// The three steps above in one launch for a batch of at most one token tile (a decode step): the membership masks
// stay in LDS, the expert offsets come from a workgroup-wide scan (two experts per lane), and every output is the
// integer the general path writes.
// Body of the one-tile permutation, by every thread of a workgroup of at least 256: a (token, choice) pair per thread
// where the work is per pair, and one scan whose lanes each own two experts (rows and tiles ride in one integer: at most
// 4096 of either), a wave at a time with one barrier between. Bound by latency: a serial loop over a token's choices and
// a workgroup-wide scan of sixteen barriers made this 9 of 14 us of a decode step's routing. s_idx [T * k] holds the
// winners already when `idx_in_lds`; the routing weights come from `prob_src` (global or LDS).
__device__ __forceinline__ void ix_moe_permute_tile_body(const int* __restrict__ topk_idx, const float* prob_src, int T,
                                                         int E, int k, int BM, int max_tiles, int* __restrict__ counts,
                                                         int* __restrict__ offsets, int* __restrict__ sorted_token,
                                                         float* __restrict__ permuted_prob,
                                                         int* __restrict__ combine_rows, int* __restrict__ meta,
                                                         int* s_idx, uint32_t* s_mask, int* s_off, int* s_sums,
                                                         bool idx_in_lds) {
  static_assert(IX_MOE_TILE_T * IX_MOE_KMAX <= 0xffff && IX_MOE_EMAX <= 512, "rows and tiles in 16 bits each");
  const int tid = threadIdx.x, nthreads = blockDim.x;
  const bool scans = tid < 256;
  for (int i = tid; i < E * 8; i += nthreads) s_mask[i] = 0u;
  if (!idx_in_lds)
    for (int i = tid; i < T * k; i += nthreads) s_idx[i] = topk_idx[i];
  __syncthreads();
  for (int i = tid; i < T * k; i += nthreads) {
    const int t = i / k;
    atomicOr(&s_mask[s_idx[i] * 8 + (t >> 5)], 1u << (t & 31));
  }
  __syncthreads();
  // lane owns experts 2 tid and 2 tid + 1
  int c[2] = {0, 0}, tl[2] = {0, 0}, own = 0, upto = 0;
  if (scans) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = 2 * tid + h;
      if (e < E) {
#pragma unroll
        for (int w = 0; w < 8; ++w) c[h] += __popc(s_mask[e * 8 + w]);
      }
      tl[h] = (c[h] + BM - 1) / BM;
    }
    own = (c[0] + c[1]) | ((tl[0] + tl[1]) << 16);
    upto = ix_wave_scan(own);
    if ((tid & 63) == 63) s_sums[tid >> 6] = upto;
  }
  __syncthreads();
  if (scans) {
    for (int w = 0; w < (tid >> 6); ++w) upto += s_sums[w];
    int row0 = (upto - own) & 0xffff;  // rows before expert 2 tid
    int tile0 = (upto - own) >> 16;
    int* tile_expert = meta + 1;
    int* tile_row0 = tile_expert + max_tiles;
    int* tile_nrows = tile_row0 + max_tiles;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = 2 * tid + h;
      if (e < E) {
        s_off[e] = row0;
        counts[e] = c[h];
        offsets[e] = row0;
        int nt = tile0;
        for (int r0 = 0; r0 < c[h] && nt < max_tiles; r0 += BM, ++nt) {
          tile_expert[nt] = e;
          tile_row0[nt] = row0 + r0;
          tile_nrows[nt] = min(BM, c[h] - r0);
        }
      }
      row0 += c[h];
      tile0 += tl[h];
    }
    if (tid == 255) {
      offsets[E] = upto & 0xffff;
      meta[0] = min(upto >> 16, max_tiles);
    }
  }
  __syncthreads();
  for (int i = tid; i < T * k; i += nthreads) {
    const int t = i / k, e = s_idx[i];
    int local = __popc(s_mask[e * 8 + (t >> 5)] & ((1u << (t & 31)) - 1u));
    for (int w = 0; w < (t >> 5); ++w) local += __popc(s_mask[e * 8 + w]);
    int rank = 0;
    for (int j2 = 0; j2 < k; ++j2) rank += (s_idx[t * k + j2] < e);
    const int pos = s_off[e] + local;
    sorted_token[pos] = t;
    permuted_prob[pos] = prob_src[i];
    combine_rows[t * k + rank] = pos;
  }
}

__global__ __launch_bounds__(256) void k_moe_permute_one_tile(const int* __restrict__ topk_idx,
                                                              const float* __restrict__ topk_prob, int T, int E,
                                                              int k, int BM, int max_tiles, int* __restrict__ counts,
                                                              int* __restrict__ offsets,
                                                              int* __restrict__ sorted_token,
                                                              float* __restrict__ permuted_prob,
                                                              int* __restrict__ combine_rows, int* __restrict__ meta) {
  __shared__ int s_idx[IX_MOE_TILE_T * IX_MOE_KMAX];
  __shared__ uint32_t s_mask[IX_MOE_EMAX * 8];
  __shared__ int s_off[IX_MOE_EMAX + 1];
  __shared__ int s_sums[4];
  ix_moe_permute_tile_body(topk_idx, topk_prob, T, E, k, BM, max_tiles, counts, offsets, sorted_token, permuted_prob,
                           combine_rows, meta, s_idx, s_mask, s_off, s_sums, false);
}

// Router and permutation of a batch of at most one token tile (a decode step) in ONE launch: a workgroup of 1024
// threads routes 64 tokens at a time (16 lanes each, ix_moe_route_row16: the function of k_moe_router_row16), keeps the
// winners in LDS, and goes straight on to the one-tile permutation above. Same integers and same weights as
// ix_moe_router_topk followed by ix_moe_permute; two launches and about ten microseconds of launch latency less.
__global__ __launch_bounds__(1024) void k_moe_route_one_tile(const float* __restrict__ logits, long ld, int T, int E,
                                                             int k, int mode, float scaling, int BM, int max_tiles,
                                                             int* __restrict__ topk_idx, float* __restrict__ topk_prob,
                                                             int* __restrict__ counts, int* __restrict__ offsets,
                                                             int* __restrict__ sorted_token,
                                                             float* __restrict__ permuted_prob,
                                                             int* __restrict__ combine_rows, int* __restrict__ meta) {
  __shared__ int s_idx[IX_MOE_TILE_T * IX_MOE_KMAX];
  __shared__ float s_prob[IX_MOE_TILE_T * IX_MOE_KMAX];
  __shared__ uint32_t s_mask[128 * 8];
  __shared__ int s_off[128 + 1];
  __shared__ int s_sums[4];
  for (int t0 = 0; t0 < T; t0 += 64) {
    const int t = t0 + (int)(threadIdx.x >> 4);
    if (t < T)
      ix_moe_route_row16(logits, ld, t, threadIdx.x & 15, E, k, mode, scaling, topk_idx, topk_prob, nullptr, nullptr,
                         s_idx, s_prob);
  }
  // (the body's first barrier publishes s_idx and s_prob)
  ix_moe_permute_tile_body(topk_idx, s_prob, T, E, k, BM, max_tiles, counts, offsets, sorted_token, permuted_prob,
                           combine_rows, meta, s_idx, s_mask, s_off, s_sums, true);
}

// Block map for rows that are ALREADY grouped by expert (the caller holds tokens_per_expert, e.g. a dispatcher's
// output): exclusive scan of the counts, then every expert writes its own row tiles. One workgroup, integer only.
// The counts live on the device, so the host cannot check them against the size of the row buffers: the kernel
// itself keeps every tile inside [0, rows) -- an expert's count is cut to what is left of `rows` after the experts
// before it (counts that add up to more than `rows` lose their tail instead of reaching past the buffers).
template <typename TI>
__global__ __launch_bounds__(256) void k_moe_block_map(const TI* __restrict__ counts_in, int E, int BM, int max_tiles,
                                                       IxMoeTall tall, int rows, int* __restrict__ offsets,
                                                       int* __restrict__ meta) {
  __shared__ int s_rows[256], s_cnt[IX_MOE_EMAX], s_off[IX_MOE_EMAX], s_toff[IX_MOE_EMAX], s_rows_per_tile;
  static_assert(IX_MOE_EMAX == 2 * 256, "a thread owns two experts");
  const int tid = threadIdx.x;
  int c[2];  // thread owns experts 2 tid and 2 tid + 1
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int e = 2 * tid + h;
    const long want = e < E ? (long)counts_in[e] : 0;
    c[h] = (int)(want < 0 ? 0 : (want > rows ? rows : want));
  }
  s_rows[tid] = min(c[0] + c[1], rows);  // a partial sum never needs to exceed `rows`: no overflow for any counts
  __syncthreads();
  for (int d = 1; d < 256; d <<= 1) {
    const int a = tid >= d ? s_rows[tid - d] : 0;
    __syncthreads();
    s_rows[tid] = min(s_rows[tid] + a, rows);
    __syncthreads();
  }
  // Saturating adds are associative for non-negative terms: s_rows[tid] = min(rows, sum of the counts up to this lane).
  const int before = tid > 0 ? s_rows[tid - 1] : 0;
  c[0] = min(c[0], rows - before);
  c[1] = min(c[1], rows - before - c[0]);
  s_cnt[2 * tid] = c[0];
  s_cnt[2 * tid + 1] = c[1];
  __syncthreads();
  if (tid < 64) {
    const int r = ix_moe_scan_experts(s_cnt, E, BM, max_tiles, tall, s_off, s_toff, true, offsets, meta);
    if (tid == 0) s_rows_per_tile = r;
  }
  __syncthreads();
  ix_moe_write_map(s_cnt, s_off, s_toff, E, s_rows_per_tile, BM, max_tiles, tall, offsets, meta);
}

static IxMoeTall ix_moe_tall(long low, int* meta, long max_tiles, long Hd, long F) {
  return {meta, (int)max_tiles, low == 160 ? IX_MOE_US_160 : IX_MOE_US_192, (int)(F / 128), (int)(Hd / IX_BK),
          (int)(Hd / 256), (int)(F / IX_BK)};
}

static int ix_moe_block_map_launch(const void* counts, int counts_i64, long E, long BM, long rows, int* offsets, int* tile_meta,
                                   long max_tiles, const IxMoeTall& tall, void* stream) {
  if (!counts || !tile_meta || E <= 0 || BM <= 0 || max_tiles <= 0 || rows < 0) return IX_ERR_ARG;
  if (E > IX_MOE_EMAX || rows > 0x3fffffffL) return IX_DECLINED;  // two clamped counts are added in an int
  hipStream_t st = (hipStream_t)stream;
  if (counts_i64)
    hipLaunchKernelGGL(k_moe_block_map<long>, dim3(1), dim3(256), 0, st, (const long*)counts, (int)E, (int)BM,
                       (int)max_tiles, tall, (int)rows, offsets, tile_meta);
  else
    hipLaunchKernelGGL(k_moe_block_map<int>, dim3(1), dim3(256), 0, st, (const int*)counts, (int)E, (int)BM,
                       (int)max_tiles, tall, (int)rows, offsets, tile_meta);
  return ix_launch_status();
}

extern "C" int ix_moe_block_map(const void* counts, int counts_i64, long E, long BM, long rows, int* offsets,
                                int* tile_meta, long max_tiles, void* stream) {
  return ix_moe_block_map_launch(counts, counts_i64, E, BM, rows, offsets, tile_meta, max_tiles, IxMoeTall{}, stream);
}

extern "C" int ix_moe_block_map_by_counts(const void* counts, int counts_i64, long E, long low, long Hd, long F, long rows,
                                          int* offsets, int* meta_low, long max_low, int* meta_tall, long max_tall,
                                          void* stream) {
  if (!meta_tall || max_tall <= 0 || Hd < 256 || F < 128 || (low != 160 && low != 192)) return IX_ERR_ARG;
  return ix_moe_block_map_launch(counts, counts_i64, E, low, rows, offsets, meta_low, max_low,
                                 ix_moe_tall(low, meta_tall, max_tall, Hd, F), stream);
}

extern "C" long ix_moe_max_tiles(long T, long k, long E, long BM) {
  if (T < 0 || k <= 0 || E <= 0 || BM <= 0) return 0;
  return (T * k + BM - 1) / BM + E;
}

extern "C" size_t ix_moe_permute_scratch_ints(long T, long E) {
  if (T < 0 || E <= 0) return 0;
  const long ntiles = (T + IX_MOE_TILE_T - 1) / IX_MOE_TILE_T;
  return (size_t)(2 * ntiles * E);
}

// Rows per tile of the ring kernels, from the mean rows per expert. Measured (E = 128, Hd = 2048, F = 768, top-8; us fc1 + fc2
// with tiles of 32 x 256 / 128 x 128 / 256 x 256): 128 tokens 221 / 221 / 237, 256 223 / 224 / 238, 400 246 / 233 / 242, 512
// 260 / 233 / 245, 700 289 / 240 / 250, 1000 328 / 253 / 253, 1500 - / 272 / 272, 2000 - / 326 / 276. 128-row tiles go with
// 128-column tiles (128 x 256: 256 at 700 tokens).
extern "C" int ix_moe_pick_bm(long T, long k, long E) {
  const long rows = T * k, e = E > 0 ? E : 1;
  return rows >= 88 * e ? 256 : (rows >= 20 * e ? 128 : 32);
}

// The same when fragment-packed copies of the matrices are at hand: the streaming kernels as long as every touched expert's
// weights are the traffic. Measured (us fc1 + fc2 with streamed tiles of 32 / 64 rows, ring 128 x 128 / 256 x 256): 64 tokens
// 176 / 177 / 219 / 242, 256 186 / 186 / 227 / 239, 512 282 / 222 / 235 / 248, 700 367 / 246 / 241 / 253, 1000 - / 366 / 254 /
// 267.
extern "C" int ix_moe_pick_bm_packed(long T, long k, long E) {
  const long rows = T * k, e = E > 0 ? E : 1;
  return rows >= 40 * e ? ix_moe_pick_bm(T, k, E) : (rows >= 16 * e ? 64 : 32);
}

// The same with the layer's sizes at hand: bands of 96, 160 and 192 rows (ix_moe_bands.h). From 24 rows per expert on (with or
// without packed matrices) the lowest in which mean + 3 sqrt(mean) rows fit, so that even routing gives every expert one tile;
// 256 from 155 on; from 240 to 400, where even routing takes two tiles of 160 or 192, these or 256 as the counts say (IxMoeTall). us
// fc1 + fc2 (E = 128, Hd = 2048, F = 768, top-8; routing even / four experts 2 to 4 times as popular / in every token's choice):
//   rows per expert   ring 128 x 128     256 rows            96                 160                192
//     28              235 / 246 / 246                        205 / 229 / 226    206 / 238 / 241
//     46              245 / 251 / 260                        214 / 237 / 239    216 / 252 / 246
//     70              259 / 262 / 276                        227 / 248 / 259    232 / 264 / 268
//     82              262 / 268 / 282                        257 / 256 / 287    234 / 268 / 271
//     106                                268 / 308 / 308                        246 / 272 / 288    250 / 284 / 291
//     124                                275 / 312 / 316                        250 / 279 / 313    254 / 289 / 301
//     133                                278 / 314 / 321                        292 / 286 / 323    256 / 295 / 307
//     160                                281 / 326 / 330                        322 / 286 / 316    305 / 303 / 341
//     241                                350 / 358 / 405                        385 / 419 / 378    419 / 414 / 374
//     277                                485 / 368 / 419                        399 / 468 / 443    428 / 474 / 389
//     331                                506 / 497 / 452                        525 / 482 / 530    485 / 523 / 487
// Over sixteen other layers of 16 to 256 experts a band of the mean is 6 % faster than the other tile in the geometric mean
// below 155 rows, the worst point 13 % slower. From 240 to 400 one of the mean is as often slower as faster (from 240 to
// 280 rows 8 % faster, 21 % and 4 % slower for the three routings, the worst point 32 %); chosen by the counts it is 5 %
// faster, the worst point 5 % slower. Both maps' launches cost 3 to 8 us more than one's.
// Not for two turns of workgroups or fewer (e F / 128 tiles): one expert that needs a second tile adds a third (32 experts
// of 2048 x 2048, 80 rows each, even / hot: 197 / 207 us in rings, 187 / 233 in bands). And not in place of the packed
// streams where these are long: us stream / 96 rows at 32 rows per expert, F = 768 (E = 128, 256) 225 / 204 and 456 / 406,
// F = 1024 (96) 332 / 294, F = 1536 (48 and 64) 166 / 187 and 411 / 412, F = 2048 (64) 269 / 286.
static bool ix_moe_bands_pay(long rows, long E, long Hd, long F) {
  return ix_moe_bands_fit(rows, Hd, F) && E * (F / 128) > 2 * IX_STREAM_WORKGROUPS;
}

extern "C" int ix_moe_pick_bm_shape(long T, long k, long E, long Hd, long F, int packed) {
  const long rows = T * k, e = E > 0 ? E : 1, mean = rows / e;
  const bool streams = packed && rows < 40 * e && F >= 1536;
  if (!streams && mean >= 24 && mean < 155 && ix_moe_bands_pay(rows, e, Hd, F)) return mean < 71 ? 96 : (mean < 127 ? 160 : 192);
  return packed ? ix_moe_pick_bm_packed(T, k, E) : ix_moe_pick_bm(T, k, E);
}

extern "C" int ix_moe_pick_low_bm(long T, long k, long E, long Hd, long F) {
  const long rows = T * k, e = E > 0 ? E : 1, mean = rows / e;
  if (mean < 240 || mean >= 400 || T <= IX_MOE_TILE_T || !ix_moe_bands_pay(rows, e, Hd, F)) return 0;
  return mean < 290 ? 160 : 192;
}

static int ix_moe_permute_launch(const int* topk_idx, const float* topk_prob, long T, long E, long k, long BM, int* counts,
                                 int* offsets, int* sorted_token, float* permuted_prob, int* combine_rows, int* tile_meta,
                                 long max_tiles, const IxMoeTall& tall, int* scratch, void* stream) {
  if (!topk_idx || !topk_prob || !counts || !offsets || !sorted_token || !permuted_prob || !combine_rows ||
      !tile_meta || !scratch)
    return IX_ERR_ARG;
  if (T < 0 || E <= 0 || k <= 0 || k > IX_MOE_KMAX || BM <= 0) return IX_ERR_ARG;
  if (E > IX_MOE_EMAX) return IX_DECLINED;
  if (max_tiles < ix_moe_max_tiles(T, k, E, BM)) return IX_ERR_ARG;
  if (T * k > 0x7fffffffL) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  const long ntiles = (T + IX_MOE_TILE_T - 1) / IX_MOE_TILE_T;
  if (ntiles == 1) {
    hipLaunchKernelGGL(k_moe_permute_one_tile, dim3(1), dim3(256), 0, st, topk_idx, topk_prob, (int)T, (int)E, (int)k,
                       (int)BM, (int)max_tiles, counts, offsets, sorted_token, permuted_prob, combine_rows, tile_meta);
    return ix_launch_status();
  }
  int* tile_counts = scratch;
  int* tile_base = scratch + ntiles * E;
  if (ntiles > 0)
    hipLaunchKernelGGL(k_moe_tile_counts, dim3((unsigned)ntiles), dim3(256), 0, st, topk_idx, (int)T, (int)E, (int)k,
                       tile_counts);
  if (ntiles > 0 && ntiles <= IX_MOE_FEW_TILES && ntiles * E <= IX_MOE_FEW_COUNTS) {
    hipLaunchKernelGGL(k_moe_offsets_scatter, dim3((unsigned)ntiles), dim3(1024), 0, st, topk_idx, topk_prob, (int)T, (int)E,
                       (int)k, (int)ntiles, (int)BM, (int)max_tiles, tall, tile_counts, counts, offsets, tile_meta,
                       sorted_token, permuted_prob, combine_rows);
    return ix_launch_status();
  }
  hipLaunchKernelGGL(k_moe_tile_prefix, dim3((unsigned)((E + 3) / 4)), dim3(256), 0, st, tile_counts, (int)ntiles, (int)E,
                     tile_base, counts);
  hipLaunchKernelGGL(k_moe_offsets, dim3(1), dim3(256), 0, st, (int)E, (int)BM, (int)max_tiles, tall, counts, offsets,
                     tile_meta);
  if (ntiles > 0)
    hipLaunchKernelGGL(k_moe_scatter, dim3((unsigned)ntiles), dim3(1024), 0, st, topk_idx, topk_prob, (int)T, (int)E,
                       (int)k, tile_base, offsets, sorted_token, permuted_prob, combine_rows);
  return ix_launch_status();
}

extern "C" int ix_moe_permute(const int* topk_idx, const float* topk_prob, long T, long E, long k, long BM,
                              int* counts, int* offsets, int* sorted_token, float* permuted_prob,
                              int* combine_rows, int* tile_meta, long max_tiles, int* scratch, void* stream) {
  return ix_moe_permute_launch(topk_idx, topk_prob, T, E, k, BM, counts, offsets, sorted_token, permuted_prob, combine_rows,
                               tile_meta, max_tiles, IxMoeTall{}, scratch, stream);
}

extern "C" int ix_moe_permute_by_counts(const int* topk_idx, const float* topk_prob, long T, long E, long k, long low, long Hd,
                                        long F, int* counts, int* offsets, int* sorted_token, float* permuted_prob, int* combine_rows,
                                        int* meta_low, long max_low, int* meta_tall, long max_tall, int* scratch,
                                        void* stream) {
  if (!meta_tall || Hd < 256 || F < 128 || (low != 160 && low != 192)) return IX_ERR_ARG;
  if (max_tall < ix_moe_max_tiles(T, k, E, 256)) return IX_ERR_ARG;
  if (T <= IX_MOE_TILE_T) return IX_DECLINED;  // one token tile: the launch without a count table
  return ix_moe_permute_launch(topk_idx, topk_prob, T, E, k, low, counts, offsets, sorted_token, permuted_prob,
                               combine_rows, meta_low, max_low, ix_moe_tall(low, meta_tall, max_tall, Hd, F), scratch, stream);
}

// ix_moe_router_topk + ix_moe_permute for a batch of at most one token tile (T <= 256) and E <= 128, in one launch.
extern "C" int ix_moe_route_one_tile(const float* logits, long ld, long T, long E, long k, int mode, float scaling,
                                     long BM, int* topk_idx, float* topk_prob, int* counts, int* offsets,
                                     int* sorted_token, float* permuted_prob, int* combine_rows, int* tile_meta,
                                     long max_tiles, void* stream) {
  if (!logits || !topk_idx || !topk_prob || !counts || !offsets || !sorted_token || !permuted_prob || !combine_rows ||
      !tile_meta)
    return IX_ERR_ARG;
  if (T < 0 || E <= 0 || k <= 0 || BM <= 0 || ld < E) return IX_ERR_ARG;
  if (mode != 0 && mode != 1) return IX_ERR_ARG;
  if (k > E || k > IX_MOE_KMAX || (k & (k - 1)) != 0) return IX_DECLINED;  // as the router
  if (T > IX_MOE_TILE_T || E > 128) return IX_DECLINED;                    // one token tile, 16 lanes per token
  if (max_tiles < ix_moe_max_tiles(T, k, E, BM)) return IX_ERR_ARG;
  hipLaunchKernelGGL(k_moe_route_one_tile, dim3(1), dim3(1024), 0, (hipStream_t)stream, logits, ld, (int)T, (int)E, (int)k,
                     mode, scaling, (int)BM, (int)max_tiles, topk_idx, topk_prob, counts, offsets, sorted_token,
                     permuted_prob, combine_rows, tile_meta);
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// The permutation for callers that cannot allocate (code under graph capture, serving loops, harnesses that forbid
// it): the two integer tables ix_moe_permute takes as `scratch` live in a file-scope device array instead. Every GPU
// the library runs on holds its own copy of the array, at its own address, until the process ends; the address is
// resolved once per device, with that device current, on the first call there. Kernels receive that address as an
// argument, exactly as they receive the caller's workspace in ix_moe_permute. Both tables are fully rewritten by
// every call before they are read (k_moe_tile_counts writes [ntiles, E], k_moe_tile_prefix writes the bases), so nothing
// has to start at zero; two calls that overlap on one GPU share the array and race.
#define IX_MOE_STATIC_SCRATCH_INTS (256 * 1024)  // 1 MiB: 2 * ceil(T / 256) * E ints, e.g. 262,144 tokens at E = 128
#define IX_MAX_DEVICES 64
static __device__ __align__(256) int ix_moe_static_scratch[IX_MOE_STATIC_SCRATCH_INTS];
static int* volatile ix_moe_static_scratch_ptr[IX_MAX_DEVICES];  // per device, 0 = not resolved yet

static int ix_moe_static_scratch_for_current_device(int** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= IX_MAX_DEVICES) return IX_ERR_LAUNCH;
  int* p = ix_moe_static_scratch_ptr[dev];
  if (!p) {
    // Two threads resolving at once store the same address: the lookup has no side effect on the array.
    void* sym = nullptr;
    if (hipGetSymbolAddress(&sym, HIP_SYMBOL(ix_moe_static_scratch)) != hipSuccess || !sym) return IX_ERR_LAUNCH;
    p = static_cast<int*>(sym);
    ix_moe_static_scratch_ptr[dev] = p;
  }
  *out = p;
  return IX_OK;
}

extern "C" size_t ix_moe_permute_static_max_ints(void) { return (size_t)IX_MOE_STATIC_SCRATCH_INTS; }

// Set-up call: resolves the array's address on the current device, so that a caller can take the one runtime lookup
// out of the region where it may make no such call (a stream capture). Launches nothing; may be called again.
extern "C" int ix_moe_permute_static_init(void) {
  int* scratch = nullptr;
  return ix_moe_static_scratch_for_current_device(&scratch);
}

extern "C" int ix_moe_permute_static(const int* topk_idx, const float* topk_prob, long T, long E, long k, long BM,
                                     int* counts, int* offsets, int* sorted_token, float* permuted_prob,
                                     int* combine_rows, int* tile_meta, long max_tiles, void* stream) {
  if (T < 0 || E <= 0) return IX_ERR_ARG;
  if (ix_moe_permute_scratch_ints(T, E) > (size_t)IX_MOE_STATIC_SCRATCH_INTS) return IX_ERR_SIZE;
  int* scratch = nullptr;
  const int rc = ix_moe_static_scratch_for_current_device(&scratch);
  if (rc != IX_OK) return rc;
  return ix_moe_permute(topk_idx, topk_prob, T, E, k, BM, counts, offsets, sorted_token, permuted_prob, combine_rows,
                        tile_meta, max_tiles, scratch, stream);
}

// ---------------------------------------------------------------------------------------------
// Grouped GEMMs over the block map. A workgroup past the device-side tile count exits at once,
// so the host never reads the routing back.
//
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM* WN * 64) void k_moe_fc1_glu(const bf16_t* __restrict__ x, long ldx, int T,
                                                             const int* __restrict__ sorted_token,
                                                             const float* __restrict__ permuted_prob,
                                                             const bf16_t* __restrict__ W1,
                                                             const int* __restrict__ meta, int max_tiles,
                                                             bf16_t* __restrict__ inter, int Hd, int F, int nb_n) {
  using Cfg = IxGemmCfg<BM, BN, WM, WN>;
  static_assert(Cfg::NI % 2 == 0, "a wave must hold gate tiles and their up tiles");
  constexpr int NP = Cfg::NI / 2;  // (gate, up) pairs of 32 columns per wave
  extern __shared__ __align__(16) char ix_lds[];
  int mt, nt;
  if (!ix_moe_tile_of_block(blockIdx.x, meta[0], nb_n, &mt, &nt)) return;
  const int e = meta[1 + mt];
  const long row0 = meta[1 + max_tiles + mt];
  const int nrows = meta[1 + 2 * max_tiles + mt];
  const int n0h = nt * (BN / 2);

  // activations: gathered token rows of x; weights: the expert's [2F, Hd] fc1 matrix with the
  // tile's rows interleaved so that each wave holds NP gate tiles (ni < NP) and their up tiles (ni >= NP):
  // tile row r -> wave r / TN, block b = (r % TN) / 32, half b / NP, column n0h + 32 * NP * wave + 32 * (b % NP) + r % 32.
  const ix_rsrc_t x_rsrc = ix_make_rsrc(x, (uint32_t)(((long)(T - 1) * ldx + Hd) * 2));
  const ix_rsrc_t w_rsrc = ix_make_rsrc(W1 + (long)e * 2 * F * Hd, (uint32_t)((long)2 * F * Hd * 2));
  auto x_row = [&](int r) -> uint32_t {
    return (r < nrows) ? (uint32_t)((long)sorted_token[row0 + r] * ldx * 2) : IX_OOB;
  };
  auto w_row = [&](int r) -> uint32_t {
    const int b = (r % Cfg::TN) >> 5;
    const int col = n0h + (r / Cfg::TN) * (32 * NP) + (b % NP) * 32 + (r & 31);
    return (col < F) ? (uint32_t)(((long)(b / NP) * F + col) * Hd * 2) : IX_OOB;
  };

  ix_f32x16 acc[Cfg::MI][Cfg::NI];
  ix_acc_zero<Cfg>(acc);
  ix_gemm_mainloop<Cfg>(x_rsrc, x_row, w_rsrc, w_row, Hd, ix_lds, acc);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  // the wave's 32 columns all exist and rows are 16-byte aligned: two half-waves join their column blocks into
  // 16-byte stores (same values, same places)
  // the same for every wave of the workgroup (a barrier depends on it): the whole tile's columns exist
  const bool wide = n0h + BN / 2 <= F && (F % 8 == 0) && (reinterpret_cast<uintptr_t>(inter) % 16 == 0);
  // late zero-fills of the ring by other waves' past-the-end fetches must not land on the store buffers
  if (wide) __syncthreads();
  char* buf = ix_lds + wave * ix_store_block32_lds_bytes<2 * NP>();
  if constexpr (Cfg::MI * Cfg::NI == 16) asm volatile("s_nop 15\n\ts_nop 15");  // matrix pipeline drained before the
                                                                                  // accumulation registers are read by hand
  // bf16(gate), bf16(up) -> s = bf16(silu(gate)) -> h = bf16(s * up) -> bf16(h * prob), two columns at a time so that
  // each rounding is one hardware pack-convert for the pair (round to nearest even; a NaN stays a NaN).
  auto chain2 = [&](float g0, float g1, float u0, float u1, float prob) -> uint32_t {
    float gate0, gate1, up0, up1, s0, s1, h0, h1;
    ix_rbf2_hw(g0, g1, gate0, gate1);
    ix_rbf2_hw(u0, u1, up0, up1);
    ix_rbf2_hw(ix_silu_div(gate0), ix_silu_div(gate1), s0, s1);
    ix_rbf2_hw(s0 * up0, s1 * up1, h0, h1);
    return ix_pack_bf2_hw(h0 * prob, h1 * prob);
  };
  ix_static_for<0, Cfg::MI>([&](auto mic) {
    constexpr int mi = decltype(mic)::value;
    const int r = wm * Cfg::TM + mi * 32 + (lane & 31);
    const bool live = r < nrows;  // the same for the two lanes that share a row
    const long m = row0 + (live ? r : 0);
    const float prob = live ? permuted_prob[m] : 0.0f;
    constexpr bool AG = Cfg::MI * Cfg::NI == 16;
    if (wide) {
      uint4 pieces[2 * NP];
      ix_static_for<0, NP>([&](auto cbc) {
        constexpr int cb = decltype(cbc)::value;  // gate block cb, up block NP + cb
        float g16[16], u16[16];
        ix_acc_read16<AG>(acc[mi][cb], g16);
        ix_acc_read16<AG>(acc[mi][NP + cb], u16);
        auto G = [&](int i) { return g16[i]; };
        auto U = [&](int i) { return u16[i]; };
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          uint2 pk[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int q = 2 * p + h;
            pk[h].x = chain2(G(q * 4), G(q * 4 + 1), U(q * 4), U(q * 4 + 1), prob);
            pk[h].y = chain2(G(q * 4 + 2), G(q * 4 + 3), U(q * 4 + 2), U(q * 4 + 3), prob);
          }
          pieces[cb * 2 + p] = ix_join_halves(pk[0], pk[1]);
        }
      });
      const int first = wm * Cfg::TM + mi * 32;  // whole rows of the wave's 32 NP columns per store instruction
      ix_store_block32_via_lds<2 * NP>(buf, pieces, inter + (row0 + first) * F + n0h + wn * (32 * NP), F,
                                       min(32, nrows - first));
      return;
    }
    if (!live) return;
    ix_static_for<0, NP>([&](auto cbc) {
      constexpr int cb = decltype(cbc)::value;
      const int c0 = n0h + wn * (32 * NP) + cb * 32;
      auto G = [&](int i) { return ix_acc_read<AG>(acc[mi][cb], i); };
      auto U = [&](int i) { return ix_acc_read<AG>(acc[mi][NP + cb], i); };
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = c0 + ix_acc_row(q * 4, lane);
        const int valid = min(4, F - col);
        if (valid <= 0) continue;
        const uint32_t lo = chain2(G(q * 4), G(q * 4 + 1), U(q * 4), U(q * 4 + 1), prob);
        const uint32_t hi = chain2(G(q * 4 + 2), G(q * 4 + 3), U(q * 4 + 2), U(q * 4 + 3), prob);
        bf16_t* dst = inter + m * F + col;
        if (valid >= 4) {
          *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);  // col % 4 == 0, F % 8 == 0, inter 16-byte aligned
        } else {
          if (valid > 0) dst[0] = (bf16_t)(lo & 0xffffu);
          if (valid > 1) dst[1] = (bf16_t)(lo >> 16);
          if (valid > 2) dst[2] = (bf16_t)(hi & 0xffffu);
        }
      }
    });
  });
}

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM* WN * 64) void k_moe_fc2(const bf16_t* __restrict__ inter,
                                                         const bf16_t* __restrict__ W2,
                                                         const int* __restrict__ meta, int max_tiles,
                                                         bf16_t* __restrict__ out, int Hd, int F, int nb_n) {
  using Cfg = IxGemmCfg<BM, BN, WM, WN>;
  extern __shared__ __align__(16) char ix_lds[];
  int mt, nt;
  if (!ix_moe_tile_of_block(blockIdx.x, meta[0], nb_n, &mt, &nt)) return;
  const int e = meta[1 + mt];
  const long row0 = meta[1 + max_tiles + mt];
  const int nrows = meta[1 + 2 * max_tiles + mt];
  const long n0 = (long)nt * BN;
  const int n_valid = (int)min((long)BN, (long)Hd - n0);

  const ix_rsrc_t x_rsrc = ix_make_rsrc(inter + row0 * F, (uint32_t)((long)nrows * F * 2));
  const ix_rsrc_t w_rsrc = ix_make_rsrc(W2 + ((long)e * Hd + n0) * F, (uint32_t)((long)n_valid * F * 2));
  auto x_row = [&](int r) -> uint32_t { return (r < nrows) ? (uint32_t)(r * F * 2) : IX_OOB; };
  auto w_row = [&](int r) -> uint32_t { return (r < n_valid) ? (uint32_t)(r * F * 2) : IX_OOB; };

  ix_f32x16 acc[Cfg::MI][Cfg::NI];
  ix_acc_zero<Cfg>(acc);
  ix_gemm_mainloop<Cfg>(x_rsrc, x_row, w_rsrc, w_row, F, ix_lds, acc);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const bool wide = n_valid == BN && (Hd % 8 == 0) && (reinterpret_cast<uintptr_t>(out) % 16 == 0);
  constexpr bool AG = Cfg::MI * Cfg::NI == 16;
  if constexpr (AG) asm volatile("s_nop 15\n\ts_nop 15");
  // late zero-fills of the ring by other waves' past-the-end fetches must not land on the store buffers
  if (wide) __syncthreads();
  constexpr int NPIECE = Cfg::NI * 2;
  char* buf = ix_lds + wave * ix_store_block32_lds_bytes<NPIECE>();
  ix_static_for<0, Cfg::MI>([&](auto mic) {
    constexpr int mi = decltype(mic)::value;
    const int r = wm * Cfg::TM + mi * 32 + (lane & 31);
    const bool live = r < nrows;  // the same for the two lanes that share a row
    const long m = row0 + r;
    if (wide) {
      uint4 pieces[NPIECE];
      ix_static_for<0, Cfg::NI>([&](auto nic) {
        constexpr int ni = decltype(nic)::value;
        float a16[16];
        ix_acc_read16<AG>(acc[mi][ni], a16);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          uint2 pk[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int q = 2 * p + h;
            pk[h].x = ix_pack_bf2_hw(a16[q * 4], a16[q * 4 + 1]);
            pk[h].y = ix_pack_bf2_hw(a16[q * 4 + 2], a16[q * 4 + 3]);
          }
          pieces[ni * 2 + p] = ix_join_halves(pk[0], pk[1]);
        }
      });
      const int first = wm * Cfg::TM + mi * 32;  // whole rows of the wave's TN columns per store instruction
      ix_store_block32_via_lds<NPIECE>(buf, pieces, out + (row0 + first) * Hd + n0 + wn * Cfg::TN, Hd,
                                       min(32, nrows - first));
      return;
    }
    if (!live) return;
    ix_static_for<0, Cfg::NI>([&](auto nic) {
      constexpr int ni = decltype(nic)::value;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const long n = n0 + wn * Cfg::TN + ni * 32 + ix_acc_row(q * 4, lane);
        const int valid = (int)min(4L, (long)Hd - n);
        if (valid <= 0) continue;
        ix_store4_bf16(out + m * Hd + n, valid, true, acc[mi][ni][q * 4], acc[mi][ni][q * 4 + 1],
                       acc[mi][ni][q * 4 + 2], acc[mi][ni][q * 4 + 3]);
      }
    });
  });
}

// ---- streaming form of the first expert GEMM (pipeline F) ------------------------------------------------------------
// The four-wave 256 x 256 tile (128 gate + 128 up columns -> 128 output columns), F a multiple of 128, Hd a multiple of
// 64 with at least NSK + 3 k-tiles. What the one-tile kernel does after its main loop -- the SwiGLU chain of 128 outputs
// per lane, two transcendentals each -- rides here on the NEXT tile's matrix instructions: when the accumulators move
// out they are kept as bf16 pairs (the chain's first rounding: gate and up, 128 registers) and each pair's chain is cut
// into eight steps of two to five instructions, one per matrix instruction of the next tile's first eight k-tiles; then,
// in four more k-tiles, the quad transposes and the stores of the plain job. (NOW > 0 sends the first NOW of the wave's four
// 32-token blocks through the chain at once instead: fewer registers, less hidden.) Same operations in the same order on
// every element as chain2() of the one-tile kernel.
// Column layout: row rho = 8 g + 4 h + i of gate block cb and of up block 2 + cb is output column 32 h + 16 cb + 4 g + i
// of the wave's 64, so a lane ends up with 32 consecutive columns of its token. The permutation is applied where the
// weight rows are fetched (the tile's LDS rows are in matrix-instruction order).
// Token ids and routing weights: every thread loads its own (eight rows' ids, four tokens' weights; the index clamped to
// the last permuted row) with loads the compiler does not count (ix_load4_uncounted), issued in the third-last k-tile
// -- ids of the NEXT tile, weights of the current one -- and taken into use in the second-last: the closing wait of the
// k-tile in between has retired them. A load the compiler knows about would make it wait for the whole operand stream
// at the first use; scalar loads cost their full latency one after the other (3.6 us per tile, measured).
// Scalar registers are short here (six pointers, five descriptors, the ring's bookkeeping): the walk over the weight
// rows is one running vector register, not eight scalar offsets, which the compiler would multiply by the k-tiles of
// the unrolled loop, spill, and reload right in front of the loads that use them.
struct IxMoeFc1StreamJob {
  const bf16_t* x;
  long ldx;
  int T;
  int rows;  // permuted rows in all (T * k)
  const int* sorted_token;
  const float* permuted_prob;
  const bf16_t* W1;
  const int* meta;
  int max_tiles;
  bf16_t* inter;
  int Hd, F, nb_n;
  unsigned xcd, idx, stride;
  static constexpr int NOW = 0;                    // 32-token blocks chained while the accumulators move out (0: all deferred)
  static constexpr int NCH = 2 * (4 - NOW);        // k-tiles of deferred chains
  static constexpr int NSK = NCH + 4;              // + one k-tile of transposes and stores per 32-token block

  ix_rsrc_t nx_xr, nx_wr;
  bool has_next;
  int nx_row0, c_row0, nx_nrows, nx_n0h, c_nrows, c_n0h;
  static constexpr int DMA_IDLE = 0;  // no reloaded scalar operand in front of a load (checked in every build)
  uint32_t xvo[8];  // this thread's eight activation chunks (gathered token rows)
  uint32_t wv;      // its next weight chunk: the ring asks for chunks 0, 1, .. 7, 0, .. and w_voff() steps it on
  int w_st16, w_stA, w_stB, w_stC;  // the four steps of that walk (bytes)
  float prob[4];    // routing weights of this lane's four tokens: set for the current tile in its second-last k-tile, read
                    // when its accumulators move out and by its deferred chains during the next tile
  ix_rsrc_t p_ir;   // pending tile: descriptor of its part of inter
  uint32_t p_voff;
  uint32_t pg[4][2][8], pu[4][2][8];  // pending gate / up values of the deferred blocks, two bf16 per register
  uint32_t res[4][2][8];              // chain results, accumulator layout
  uint32_t ta[4][4], tb[4][4];
  float g0, g1, a0, a1;               // a chain in flight

  __device__ __forceinline__ void locate() {
    int mt = 0, nt = 0;
    has_next = ix_moe_tile_of_block(xcd + 8u * idx, meta[0], nb_n, &mt, &nt);
    if (!has_next) {  // no tile: no rows, and a weight descriptor without bytes (its fetches touch no memory)
      nx_row0 = nx_nrows = nx_n0h = 0;
      nx_wr = ix_make_rsrc(W1, 0u);
      return;
    }
    const long e = meta[1 + mt];
    nx_row0 = meta[1 + max_tiles + mt];
    nx_nrows = meta[1 + 2 * max_tiles + mt];
    nx_n0h = nt * 128;
    // weights: the expert's gate rows n0h .. n0h + 127 and, F rows further on, its up rows
    nx_wr = ix_make_rsrc(W1 + (e * 2 * F + nx_n0h) * Hd, (uint32_t)(((long)F + 128) * Hd * 2));
  }
  __device__ __forceinline__ uint32_t kb() const {
    return (uint32_t)(((threadIdx.x & 7) ^ ix_swz8(threadIdx.x >> 3)) * 16);  // rows 32 apart share the swizzle
  }
  // Loads for the tile after the current one (token ids of this thread's eight rows: tile row r0 + 32 j of chunk j,
  // r0 = thread / 8) and for the current one (routing weights of this lane's four tokens). In flight until take_gathers().
  uint32_t g_tok[8], g_prob[4];
  __device__ __forceinline__ void issue_gathers() {
    const int r0 = threadIdx.x >> 3, last = rows - 1;
    const int trow = (int)(threadIdx.x >> 7) * 128 + (int)(threadIdx.x & 31);  // token of accumulator block row 0
    ix_static_for<0, 8>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      g_tok[j] = ix_load4_uncounted(sorted_token, (uint32_t)min(nx_row0 + r0 + 32 * j, last) * 4u);
    });
    ix_static_for<0, 4>([&](auto mc) {
      constexpr int mi = decltype(mc)::value;
      g_prob[mi] = ix_load4_uncounted(permuted_prob, (uint32_t)min(c_row0 + trow + 32 * mi, last) * 4u);
    });
  }
  __device__ __forceinline__ void take_gathers() {
    const int r0 = threadIdx.x >> 3;
    ix_static_for<0, 8>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const uint32_t tok = ix_landed(g_tok[j]);
      // a row the tile does not have (a missing next tile has none) gets an offset outside the descriptor
      xvo[j] = (r0 + 32 * j < nx_nrows) ? tok * (uint32_t)(ldx * 2) + kb() : IX_OOB;
    });
    // rows past the tile's last got some row's weight: their products are dropped by the store's range check
    ix_static_for<0, 4>([&](auto mc) { prob[decltype(mc)::value] = __uint_as_float(ix_landed(g_prob[decltype(mc)::value])); });
  }
  __device__ __forceinline__ bool open_first() {
    xcd = blockIdx.x & 7u;
    idx = blockIdx.x >> 3;
    stride = gridDim.x >> 3;
    nx_xr = ix_make_rsrc(x, (uint32_t)(((long)(T - 1) * ldx + Hd) * 2));  // the same for every tile
    locate();
    p_ir = ix_make_rsrc(nullptr, 0u);  // the empty pending tile
    p_voff = IX_OOB;
#pragma unroll
    for (int i = 0; i < 64; ++i) pg[i >> 4][(i >> 3) & 1][i & 7] = pu[i >> 4][(i >> 3) & 1][i & 7] = res[i >> 4][(i >> 3) & 1][i & 7] = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) prob[i] = 0.0f;
    g0 = g1 = a0 = a1 = 0.0f;
    return has_next;
  }
  __device__ __forceinline__ void open_next() {  // start of the third-last k-tile
    idx += stride;
    locate();
    issue_gathers();
  }
  __device__ __forceinline__ void first_voffs() {
    {  // the first tile's rows: nothing is in flight yet, ordinary loads
      const int r0 = threadIdx.x >> 3;
      uint32_t tok[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) tok[j] = (uint32_t)sorted_token[min(nx_row0 + r0 + 32 * j, rows - 1)];
#pragma unroll
      for (int j = 0; j < 8; ++j) xvo[j] = (r0 + 32 * j < nx_nrows) ? tok[j] * (uint32_t)(ldx * 2) + kb() : IX_OOB;
    }
    // Weight tile row r0 + 32 j (chunk j of thread row r0) = wave column j / 4, block j % 4 (gate 0, gate 1, up 0, up 1),
    // matrix-instruction row r0: weight row [up: F] + 64 (j / 4) + 16 (j % 2) + lane_col(r0) of the descriptor.
    // In rows, chunk 0..7 = 0, 16, F, F + 16, 64, 80, F + 64, F + 80 (+ lane_col); the walk's steps are the differences.
    const int r0 = threadIdx.x >> 3;
    const int lane_col = 32 * ((r0 >> 2) & 1) + 4 * (r0 >> 3) + (r0 & 3);
    wv = (uint32_t)((long)lane_col * Hd * 2) + kb();
    const int row_bytes = Hd * 2;
    w_st16 = __builtin_amdgcn_readfirstlane(16 * row_bytes);
    w_stA = __builtin_amdgcn_readfirstlane((F - 16) * row_bytes);
    w_stB = __builtin_amdgcn_readfirstlane((48 - F) * row_bytes);
    w_stC = __builtin_amdgcn_readfirstlane(-(F + 80) * row_bytes);
  }
  template <int J>
  __device__ __forceinline__ uint32_t x_voff() const { return xvo[J]; }
  // The step is added by an instruction the compiler cannot hoist, or it would keep every sum of every k-tile in a
  // register of its own.
  template <int J>
  __device__ __forceinline__ uint32_t w_voff() {
    const uint32_t v = wv;
    asm volatile("v_add_u32 %0, %1, %0" : "+v"(wv) : "s"(J == 7 ? w_stC : (J == 3 ? w_stB : ((J & 1) ? w_stA : w_st16))));
    return v;
  }
  // second-last k-tile, after the current tile's last fetch through xvo: the loads of the k-tile before have retired
  __device__ __forceinline__ void turn_offsets() { take_gathers(); }
  __device__ __forceinline__ void advance() {
    c_row0 = nx_row0;
    c_nrows = nx_nrows;
    c_n0h = nx_n0h;
  }
  // bf16(gate), bf16(up) -> s = bf16(silu(gate)) -> h = bf16(s * up) -> bf16(h * prob), two columns at a time
  static __device__ __forceinline__ uint32_t chain2(float g0_, float g1_, float u0_, float u1_, float p) {
    float gate0, gate1, up0, up1, s0, s1, h0, h1;
    ix_rbf2_hw(g0_, g1_, gate0, gate1);
    ix_rbf2_hw(u0_, u1_, up0, up1);
    ix_rbf2_hw(ix_silu_div(gate0), ix_silu_div(gate1), s0, s1);
    ix_rbf2_hw(s0 * up0, s1 * up1, h0, h1);
    return ix_pack_bf2_hw(h0 * p, h1 * p);
  }
  template <typename Acc>
  __device__ __forceinline__ void drain(Acc& acc) {
    ix_static_for<0, 8>([&](auto bc) {
      constexpr int mi = decltype(bc)::value >> 1, cb = decltype(bc)::value & 1;
      float g16[16], u16[16];
      ix_acc_read16<true>(acc[mi][cb], g16);
      ix_acc_read16<true>(acc[mi][2 + cb], u16);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (mi < NOW) {
          res[mi][cb][i] = chain2(g16[2 * i], g16[2 * i + 1], u16[2 * i], u16[2 * i + 1], prob[mi]);
        } else {
          pg[mi][cb][i] = ix_pack_bf2_hw(g16[2 * i], g16[2 * i + 1]);
          pu[mi][cb][i] = ix_pack_bf2_hw(u16[2 * i], u16[2 * i + 1]);
        }
      }
      if constexpr (mi < NOW) {
        ix_pin8(res[mi][cb]);
      } else {
        ix_pin8(pg[mi][cb]);
        ix_pin8(pu[mi][cb]);
      }
    });
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // after the quad transposes a lane holds piece (lane % 4) of the four tokens of its quad
    const int r = (wave >> 1) * 128 + (lane & 28), c = (wave & 1) * 64 + 32 * (lane >> 5) + 8 * (lane & 3);
    p_ir = ix_make_rsrc(inter + (long)c_row0 * F + c_n0h, (uint32_t)(((long)(c_nrows - 1) * F + 128) * 2));
    p_voff = (uint32_t)(((long)r * F + c) * 2);
  }
  static constexpr int stores_after_p1(int s) { return s >= NCH ? 4 : 0; }
  static __device__ __forceinline__ int w_frag_row(int ni, int rho) { return ni * 32 + rho; }
  // k-tile s < NCH: the eight chains of (mi = NOW + s / 2, cb = s % 2), chain c in slots 8 c .. 8 c + 7.
  // k-tile s = NCH + mi: the 32 tokens mi: exchange stage 1 in slots 0..15, stage 2 in 16..31, stores 32..35.
  template <int I>
  __device__ __forceinline__ void micro() {
    constexpr int s = I / 64, q = I % 64;
    if constexpr (s < NCH) {
      constexpr int mi = NOW + (s >> 1), cb = s & 1, c = q >> 3, st = q & 7;
      if constexpr (st == 0) {
        g0 = __uint_as_float(pg[mi][cb][c] << 16);
        g1 = __uint_as_float(pg[mi][cb][c] & 0xffff0000u);
        a0 = (-g0) * IX_LOG2E;
        a1 = (-g1) * IX_LOG2E;
      } else if constexpr (st == 1) {
        a0 = ix_exp2(a0);
      } else if constexpr (st == 2) {
        a1 = ix_exp2(a1);
      } else if constexpr (st == 3) {
        a0 = 1.0f + a0;
        a1 = 1.0f + a1;
        a0 = __builtin_amdgcn_rcpf(a0);
      } else if constexpr (st == 4) {
        a1 = __builtin_amdgcn_rcpf(a1);
        a0 = g0 * a0;
      } else if constexpr (st == 5) {
        a1 = g1 * a1;
        ix_rbf2_hw(a0, a1, a0, a1);
      } else if constexpr (st == 6) {
        const float u0 = __uint_as_float(pu[mi][cb][c] << 16), u1 = __uint_as_float(pu[mi][cb][c] & 0xffff0000u);
        ix_rbf2_hw(a0 * u0, a1 * u1, a0, a1);
      } else {
        res[mi][cb][c] = ix_pack_bf2_hw(a0 * prob[mi], a1 * prob[mi]);
      }
    } else {
      constexpr int mi = s - NCH;
      if constexpr (q < 16) {
        // piece pi, dword d of the lane's 64 bytes: res[mi][pi / 2][4 (pi % 2) + d]; stage 1 pairs pieces (0, 1), (2, 3)
        constexpr int d = q >> 2, t = q & 3, a = t & 2;
        ta[t][d] = ix_quad_exchange<1, (t & 1) != 0>(res[mi][a >> 1][d], res[mi][a >> 1][4 + d]);
      } else if constexpr (q < 32) {
        constexpr int o = q - 16, d = o >> 2, t = o & 3, a = t & 1;
        tb[t][d] = ix_quad_exchange<2, (t & 2) != 0>(ta[a][d], ta[a + 2][d]);
      } else if constexpr (q < 36) {
        constexpr int t = q - 32;  // token t of the quad
        ix_buffer_store16<IX_STREAM_STORE_NT_FC1>(make_uint4(tb[t][0], tb[t][1], tb[t][2], tb[t][3]), p_ir,
                          p_voff == IX_OOB ? IX_OOB : p_voff + (uint32_t)((long)(mi * 32 + t) * F * 2));
      }
    }
  }
};

template <bool W_ONCE>
__global__ __launch_bounds__(256) void k_moe_fc1_glu_stream(const bf16_t* __restrict__ x, long ldx, int T, int rows,
                                                            const int* __restrict__ sorted_token,
                                                            const float* __restrict__ permuted_prob,
                                                            const bf16_t* __restrict__ W1, const int* __restrict__ meta,
                                                            int max_tiles, bf16_t* __restrict__ inter, int Hd, int F,
                                                            int nb_n) {
  using Cfg = IxGemmCfg<256, 256, 2, 2, 0, W_ONCE>;
  extern __shared__ __align__(16) char ix_lds[];
  IxMoeFc1StreamJob job;
  job.x = x;
  job.ldx = ldx;
  job.T = T;
  job.rows = rows;
  job.sorted_token = sorted_token;
  job.permuted_prob = permuted_prob;
  job.W1 = W1;
  job.meta = meta;
  job.max_tiles = max_tiles;
  job.inter = inter;
  job.Hd = Hd;
  job.F = F;
  job.nb_n = nb_n;
  ix_gemm_stream4<Cfg>(job, Hd / IX_BK, ix_lds);
}

template <int BM, int BN, int WM, int WN>
static int ix_moe_experts_launch(const bf16_t* x, long ldx, int T, long rows, const int* sorted_token,
                                 const float* permuted_prob,
                                 const bf16_t* W1, const bf16_t* W2, const int* meta, long max_tiles,
                                 bf16_t* inter, bf16_t* out, int Hd, int F, hipStream_t st) {
  using Cfg = IxGemmCfg<BM, BN, WM, WN>;
  using CfgOnce = IxGemmCfg<BM, BN, WM, WN, 0, true>;
  auto k1 = k_moe_fc1_glu<BM, BN, WM, WN>;
  auto k2 = k_moe_fc2<BM, BN, WM, WN>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)k1, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES) !=
            hipSuccess ||
        hipFuncSetAttribute((const void*)k2, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES) !=
            hipSuccess)
      return IX_ERR_LAUNCH;
    attr_set = true;
  }
  const long nb1 = (F + BN / 2 - 1) / (BN / 2);
  const long nb2 = (Hd + BN - 1) / BN;
  if (max_tiles * nb1 > 0x7fffffffL || max_tiles * nb2 > 0x7fffffffL) return IX_DECLINED;
  // Weights read past the caches (ix_dma16) while nearly every expert has one 256-row tile, i.e. each of its weight tiles
  // one reader: mean rows per expert up to 224 (max_tiles counts one tile per expert beside the full ones). us fc1 + fc2,
  // 128 experts of 2048 x 768: 512 tokens 278 -> 259, 1500 300 -> 287, 3500 335 -> 310; 4096 tokens, where half the experts
  // have a second tile, 410 -> 419.
  const bool once = rows <= 224 * (max_tiles - rows / 256);
  // 8 XCD runs of the tile order; the longest run sets the count
  bool fc1_streamed = false;
  if constexpr (BM == 256 && BN == 256 && WM == 2 && WN == 2) {
    // worth it from two tiles per workgroup up (max_tiles bounds the row tiles from above by at most one per expert)
    // (32-bit byte offsets into the permutation's arrays and into an expert's weight rows)
    if (Hd % IX_BK == 0 && Hd / IX_BK >= IxMoeFc1StreamJob::NSK + 3 && F % 128 == 0 && rows > 0 && rows < 0x20000000L &&
        ((long)F + 128) * Hd * 2 < 0x40000000L && max_tiles * nb1 >= 2 * IX_STREAM_WORKGROUPS) {
      static bool attr1_set = false;
      if (!attr1_set) {
        if (hipFuncSetAttribute((const void*)k_moe_fc1_glu_stream<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                Cfg::LDS_BYTES) != hipSuccess ||
            hipFuncSetAttribute((const void*)k_moe_fc1_glu_stream<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                Cfg::LDS_BYTES) != hipSuccess)
          return IX_ERR_LAUNCH;
        attr1_set = true;
      }
      hipLaunchKernelGGL(once ? k_moe_fc1_glu_stream<true> : k_moe_fc1_glu_stream<false>, dim3(IX_STREAM_WORKGROUPS), dim3(256), Cfg::LDS_BYTES, st, x, ldx, T,
                         (int)rows, sorted_token, permuted_prob, W1, meta, (int)max_tiles, inter, Hd, F, (int)nb1);
      fc1_streamed = true;
    }
  }
  if (!fc1_streamed)
    hipLaunchKernelGGL(k1, dim3((unsigned)(8 * ((max_tiles * nb1 + 7) / 8))), dim3(Cfg::NT), Cfg::LDS_BYTES, st, x, ldx, T,
                       sorted_token, permuted_prob, W1, meta, (int)max_tiles, inter, Hd, F, (int)nb1);
  if constexpr (BM == 256 && BN == 256 && WM == 2 && WN == 2) {
    // worth it from two tiles per workgroup up (max_tiles bounds the row tiles from above by at most one per expert)
    if (F % IX_BK == 0 && F / IX_BK >= IX_STREAM_MIN_KT && Hd % 256 == 0 && (long)Hd * 512 < 0x40000000L &&
        max_tiles * nb2 >= 2 * IX_STREAM_WORKGROUPS) {
      static bool attr2_set = false;
      if (!attr2_set) {
        if (hipFuncSetAttribute((const void*)k_moe_fc2_stream<Cfg>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                Cfg::LDS_BYTES) != hipSuccess ||
            hipFuncSetAttribute((const void*)k_moe_fc2_stream<CfgOnce>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                Cfg::LDS_BYTES) != hipSuccess)
          return IX_ERR_LAUNCH;
        attr2_set = true;
      }
      hipLaunchKernelGGL(once ? k_moe_fc2_stream<CfgOnce> : k_moe_fc2_stream<Cfg>, dim3(IX_STREAM_WORKGROUPS), dim3(256), Cfg::LDS_BYTES, st, inter, W2, meta,
                         (int)max_tiles, out, Hd, F, (int)nb2);
      return ix_launch_status();
    }
  }
  hipLaunchKernelGGL(k2, dim3((unsigned)(8 * ((max_tiles * nb2 + 7) / 8))), dim3(Cfg::NT), Cfg::LDS_BYTES, st, inter, W2, meta,
                     (int)max_tiles, out, Hd, F, (int)nb2);
  return ix_launch_status();
}

extern "C" int ix_moe_experts_tile(const void* x, long ldx, const int* sorted_token, const float* permuted_prob,
                                   const void* W1, const void* W2, const int* tile_meta, long max_tiles, long BM,
                                   long BN, void* inter, void* expert_out, long T, long rows, long Hd, long F,
                                   void* stream) {
  if (!x || !sorted_token || !permuted_prob || !W1 || !W2 || !tile_meta || !inter || !expert_out)
    return IX_ERR_ARG;
  if (T < 0 || rows < 0 || Hd <= 0 || F <= 0 || max_tiles < 0 || ldx < Hd) return IX_ERR_ARG;
  // 32-bit buffer offsets: the activation matrix, one expert's weights and one row tile must fit
  if (T * ldx * 2 >= 0x40000000L || 2 * F * Hd * 2 >= 0x40000000L || 256 * F * 2 >= 0x40000000L) return IX_DECLINED;
  if ((Hd % 8) || (F % 8) || (ldx % 8) || !ix_aligned(x, 16) || !ix_aligned(W1, 16) || !ix_aligned(W2, 16) ||
      !ix_aligned(inter, 16) || !ix_aligned(expert_out, 8))
    return IX_DECLINED;
  if (rows == 0 || max_tiles == 0) return IX_OK;
  hipStream_t st = (hipStream_t)stream;
  const bf16_t *xx = (const bf16_t*)x, *w1 = (const bf16_t*)W1, *w2 = (const bf16_t*)W2;
  bf16_t *it = (bf16_t*)inter, *eo = (bf16_t*)expert_out;
  if (BN != 256 && !(BN == 128 && BM == 128)) return IX_ERR_ARG;
  if (BN == 128)
    return ix_moe_experts_launch<128, 128, 2, 2>(xx, ldx, (int)T, rows, sorted_token, permuted_prob, w1, w2, tile_meta,
                                                 max_tiles, it, eo, (int)Hd, (int)F, st);
  if (BM == 96 || BM == 160 || BM == 192 || BM == 224) {
    if (BM != 224 && ix_moe_bands_fit(rows, Hd, F) && ix_aligned(expert_out, 16)) {
      auto bands = BM < 192 ? ix_moe_experts_bands_low : ix_moe_experts_bands_high;
      return bands((int)BM, xx, ldx, (int)T, rows, sorted_token, permuted_prob, w1, w2, tile_meta, max_tiles, it, eo, (int)Hd,
                   (int)F, st);
    }
    BM = 256;  // a taller tile holds the map's rows as well (224 rows have no kernel of their own)
  }
  switch (BM) {
    case 32:
      return ix_moe_experts_launch<32, 256, 1, 4>(xx, ldx, (int)T, rows, sorted_token, permuted_prob, w1, w2, tile_meta,
                                                  max_tiles, it, eo, (int)Hd, (int)F, st);
    case 128:
      return ix_moe_experts_launch<128, 256, 2, 4>(xx, ldx, (int)T, rows, sorted_token, permuted_prob, w1, w2, tile_meta,
                                                   max_tiles, it, eo, (int)Hd, (int)F, st);
    case 256:
      return ix_moe_experts_launch<256, 256, 2, 2>(xx, ldx, (int)T, rows, sorted_token, permuted_prob, w1, w2, tile_meta,
                                                   max_tiles, it, eo, (int)Hd, (int)F, st);
    default: return IX_ERR_ARG;
  }
}

extern "C" int ix_moe_experts(const void* x, long ldx, const int* sorted_token, const float* permuted_prob,
                              const void* W1, const void* W2, const int* tile_meta, long max_tiles, long BM,
                              void* inter, void* expert_out, long T, long rows, long Hd, long F, void* stream) {
  return ix_moe_experts_tile(x, ldx, sorted_token, permuted_prob, W1, W2, tile_meta, max_tiles, BM, 256, inter,
                             expert_out, T, rows, Hd, F, stream);
}

// ---------------------------------------------------------------------------------------------
// The grouped GEMMs of a decode step: weights streamed through registers.
//
// At decode sizes an expert has a handful of rows, the matrix pipes idle and the step is the time memory needs to
// deliver every touched expert's weights once. The ring kernels above stage weights in LDS, so a CU never has more
// than its 160 KiB in flight (one workgroup, ~100 KiB of weight bytes): about 5.1 TB/s. Here no LDS is used at all:
//   * weights are stored FRAGMENT-PACKED (ix_moe_pack_decode): per (expert, column tile, wave, k-tile) the 8 KiB a wave's
//     eight matrix instructions of that k-tile take as their A operands, in (block, step, lane) order, so that a load
//     instruction is 1 KiB of contiguous memory and a wave walks one contiguous stream;
//   * a lane keeps the fragments of the next D k-tiles in registers (D x 8 loads of 16 bytes in flight per lane, eight
//     waves per CU: up to 256 KiB of weight bytes in flight per CU), loaded past the caches where ix_streams_once says so;
//   * activations (at most 32 token rows per block, typically four live ones) come straight from memory as B operands,
//     a lane loading the 16 bytes of its own token, as far ahead as the weights; a dead token's lanes load a live row
//     and multiply zeros instead;
//   * a workgroup is ONE wave (a column tile's four waves share nothing), so that a step that touches few experts spreads
//     over the chip: one token's eight experts are 192 workgroups instead of 48 (fc1 23.3 -> 10.4 us);
//   * a block map of 64-row tiles (BM = 64) multiplies up to two blocks of 32 tokens with the same weight registers.
// Measured (E = 128, Hd = 2048, F = 768, top-8; us fc1 / fc2, four waves and default loads -> this): T = 1 23.3 / 8.3 ->
// 10.4 / 5.7; T = 64 132 / 68 -> 116 / 57 (7.0 TB/s); T = 512 (32-row tiles, experts with more rows read twice) 175 / 89 ->
// 136 / 80 (64-row tiles).
// Arithmetic is that of every other tile shape: v_mfma_f32_32x32x16_bf16, weights the A operand, K in tiles of 64, step
// s consuming k = 8 s .. 8 s + 7 (lane group 0) and 32 + 8 s .. (lane group 1), one fp32 accumulator per element, the
// epilogues of k_moe_fc1_glu / k_moe_fc2 statement for statement.
// Packed layouts (16-byte chunk index; r = lane % 32, g = lane / 32; chunk = W[row][64 kt + 32 g + 8 s .. + 7]):
//   W1f [E][F / 128][wave 4][Hd / 64][b 2][s 4][lane 64]   row = b F + 128 nt + 32 wave + r      (b: gate, up)
//   W2f [E][Hd / 256][wave 4][F / 64][b 2][s 4][lane 64]   row = 256 nt + 64 wave + 32 b + r
__global__ __launch_bounds__(256) void k_moe_pack_frag(const bf16_t* __restrict__ W, bf16_t* __restrict__ Wf,
                                                       int rows_per_expert, int K, int nb, int is_fc1, long chunks) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= chunks) return;
  const int KT = K / 64;
  const int lane = (int)(i & 63), st = (int)((i >> 6) & 3), b = (int)((i >> 8) & 1);
  long rest = i >> 9;
  const int kt = (int)(rest % KT);
  rest /= KT;
  const int w = (int)(rest & 3);
  rest >>= 2;
  const int nt = (int)(rest % nb);
  const long e = rest / nb;
  const int r = lane & 31, g = lane >> 5;
  const int row = is_fc1 ? b * (rows_per_expert / 2) + 128 * nt + 32 * w + r : 256 * nt + 64 * w + 32 * b + r;
  const uint4 v = *reinterpret_cast<const uint4*>(W + (e * rows_per_expert + row) * (long)K + 64 * kt + 32 * g + 8 * st);
  *reinterpret_cast<uint4*>(Wf + i * 8) = v;
}

// D: k-tiles of fragments a lane holds ahead of the matrix instructions. TB: blocks of 32 token rows. ONCE: weights past the
// caches.
template <int D, int TB, bool ONCE>
struct IxDecStream {
  const uint4* wp;       // this lane's first chunk of the wave's stream: k-tile kt, chunk c at wp[kt * 512 + c * 64]
  const bf16_t* xp[TB];  // this lane's token row + 32 g (a dead token's lanes point at a live row and discard what they load)
  bool live[TB];
  uint4 wreg[D][8];
  uint4 xreg[D][TB][4];
  __device__ __forceinline__ void load(int d, int kt) {
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int st = 0; st < 4; ++st) xreg[d][t][st] = *reinterpret_cast<const uint4*>(xp[t] + 64 * kt + 8 * st);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint4* p = wp + (long)kt * 512 + c * 64;
      wreg[d][c] = ONCE ? ix_load16_once(p) : *p;
    }
  }
  __device__ __forceinline__ void multiply(int d, ix_f32x16 (&a0)[TB], ix_f32x16 (&a1)[TB]) {
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        uint4 xv = xreg[d][t][st];
        if (!live[t]) xv = make_uint4(0u, 0u, 0u, 0u);  // a select, not a branch
        const ix_bf16x8 xf = *reinterpret_cast<const ix_bf16x8*>(&xv);
        a0[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const ix_bf16x8*>(&wreg[d][st]), xf, a0[t], 0, 0, 0);
        a1[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const ix_bf16x8*>(&wreg[d][4 + st]), xf, a1[t], 0, 0, 0);
      }
  }
  // The whole product of a wave: two 32 x 32 blocks per token block (weight chunks 0..3 -> a0, 4..7 -> a1) over KT_ k-tiles.
  // KT_ is a compile-time constant and the walk is straight-line code: with a loop (or any branch) the compiler's wait
  // bookkeeping falls back to "wait for every load" at the join, which would drain the D k-tiles in flight at every
  // step; in straight-line code it waits for exactly the loads a matrix instruction reads.
  template <int KT_>
  __device__ __forceinline__ void run(ix_f32x16 (&a0)[TB], ix_f32x16 (&a1)[TB]) {
    static_assert(KT_ >= D, "the ring is filled before the first multiply");
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) a0[t][i] = a1[t][i] = 0.0f;
    // sched_barrier(0): the compiler's scheduler may not move a load across it -- left alone it sinks every load down
    // to its first use (fewest live registers), which is a ring of depth zero. Loads retire in order, so the
    // activation fragments of a k-tile are requested together with its weight fragments, D k-tiles ahead: a wait for
    // k-tile kt then leaves the younger k-tiles' loads in flight.
    ix_static_for<0, D>([&](auto dc) { load(decltype(dc)::value, decltype(dc)::value); });
    __builtin_amdgcn_sched_barrier(0);
    ix_static_for<0, KT_>([&](auto kc) {
      constexpr int kt = decltype(kc)::value, d = kt % D;
      multiply(d, a0, a1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kt + D < KT_) load(d, kt + D);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
};

// unit -> (row tile, column tile, wave of the packed layout)
struct IxDecUnit {
  long e, row0, stream;  // stream: index of the unit's packed stream
  int nrows, nt, w;
  __device__ __forceinline__ bool init(const int* __restrict__ meta, int max_tiles, int nb_n) {
    int mt, u;
    if (!ix_moe_tile_of_block(blockIdx.x, meta[0], nb_n * 4, &mt, &u)) return false;
    e = meta[1 + mt];
    row0 = meta[1 + max_tiles + mt];
    nrows = meta[1 + 2 * max_tiles + mt];
    nt = u >> 2;
    w = u & 3;
    stream = (e * nb_n + nt) * 4 + w;
    return true;
  }
};

template <int D, int TB, bool ONCE, int KT>
__device__ __forceinline__ void ix_moe_fc1_dec_unit(const IxDecUnit& un, const bf16_t* __restrict__ x, long ldx,
                                                    const int* __restrict__ sorted_token,
                                                    const float* __restrict__ permuted_prob, const bf16_t* __restrict__ W1f,
                                                    bf16_t* __restrict__ inter, int F) {
  const int lane = threadIdx.x, r = lane & 31, g = lane >> 5;
  IxDecStream<D, TB, ONCE> st;
  st.wp = reinterpret_cast<const uint4*>(W1f) + un.stream * (long)KT * 512 + lane;
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    st.live[t] = 32 * t + r < un.nrows;
    st.xp[t] = x + (long)sorted_token[un.row0 + (st.live[t] ? 32 * t + r : 0)] * ldx + 32 * g;  // a tile has at least one row
  }
  ix_f32x16 ag[TB], au[TB];
  st.template run<KT>(ag, au);
  const int c0 = un.nt * 128 + un.w * 32;
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    if (!st.live[t]) continue;
    const long m = un.row0 + 32 * t + r;
    const float prob = permuted_prob[m];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int col = c0 + ix_acc_row(q * 4, lane);
      const uint32_t lo = IxMoeFc1StreamJob::chain2(ag[t][q * 4], ag[t][q * 4 + 1], au[t][q * 4], au[t][q * 4 + 1], prob);
      const uint32_t hi =
          IxMoeFc1StreamJob::chain2(ag[t][q * 4 + 2], ag[t][q * 4 + 3], au[t][q * 4 + 2], au[t][q * 4 + 3], prob);
      *reinterpret_cast<uint2*>(inter + m * F + col) = make_uint2(lo, hi);  // col % 4 == 0, F % 8 == 0, inter 16-byte aligned
    }
  }
}

template <int D, int TB, bool ONCE, int KT>
__device__ __forceinline__ void ix_moe_fc2_dec_unit(const IxDecUnit& un, const bf16_t* __restrict__ inter,
                                                    const bf16_t* __restrict__ W2f, bf16_t* __restrict__ out, int Hd, int F) {
  const int lane = threadIdx.x, r = lane & 31, g = lane >> 5;
  IxDecStream<D, TB, ONCE> st;
  st.wp = reinterpret_cast<const uint4*>(W2f) + un.stream * (long)KT * 512 + lane;
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    st.live[t] = 32 * t + r < un.nrows;
    st.xp[t] = inter + (un.row0 + (st.live[t] ? 32 * t + r : 0)) * (long)F + 32 * g;
  }
  ix_f32x16 a0[TB], a1[TB];
  st.template run<KT>(a0, a1);
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    if (!st.live[t]) continue;
    const long m = un.row0 + 32 * t + r;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long n = (long)un.nt * 256 + un.w * 64 + ix_acc_row(q * 4, lane);
      ix_store4_bf16(out + m * Hd + n, 4, true, a0[t][q * 4], a0[t][q * 4 + 1], a0[t][q * 4 + 2], a0[t][q * 4 + 3]);
      ix_store4_bf16(out + m * Hd + n + 32, 4, true, a1[t][q * 4], a1[t][q * 4 + 1], a1[t][q * 4 + 2], a1[t][q * 4 + 3]);
    }
  }
}

// BM = 32 or 64: the block map's rows per tile. Four k-tiles ahead for one block of tokens (three where a long K's addresses
// would push registers out to memory), two for two: both leave two waves per SIMD; deeper rings with one wave measured slower.
template <int KT, int BM, bool ONCE>
__global__ __launch_bounds__(64, 2) void k_moe_fc1_dec(const bf16_t* __restrict__ x, long ldx,
                                                       const int* __restrict__ sorted_token,
                                                       const float* __restrict__ permuted_prob,
                                                       const bf16_t* __restrict__ W1f, const int* __restrict__ meta,
                                                       int max_tiles, bf16_t* __restrict__ inter, int F, int nb_n) {
  IxDecUnit un;
  if (!un.init(meta, max_tiles, nb_n)) return;
  if (BM == 32 || un.nrows <= 32)
    ix_moe_fc1_dec_unit<(KT <= 32 ? 4 : 3), 1, ONCE, KT>(un, x, ldx, sorted_token, permuted_prob, W1f, inter, F);
  else
    ix_moe_fc1_dec_unit<2, 2, ONCE, KT>(un, x, ldx, sorted_token, permuted_prob, W1f, inter, F);
}

template <int KT, int BM, bool ONCE>
__global__ __launch_bounds__(64, 2) void k_moe_fc2_dec(const bf16_t* __restrict__ inter, const bf16_t* __restrict__ W2f,
                                                       const int* __restrict__ meta, int max_tiles,
                                                       bf16_t* __restrict__ out, int Hd, int F, int nb_n) {
  IxDecUnit un;
  if (!un.init(meta, max_tiles, nb_n)) return;
  if (BM == 32 || un.nrows <= 32)
    ix_moe_fc2_dec_unit<(KT <= 12 ? 4 : 3), 1, ONCE, KT>(un, inter, W2f, out, Hd, F);
  else
    ix_moe_fc2_dec_unit<2, 2, ONCE, KT>(un, inter, W2f, out, Hd, F);
}

// The k-tile counts the straight-line kernels are instantiated for (K = 64 KT).
#define IX_DEC_KTS(M) M(8) M(12) M(16) M(24) M(32) M(48) M(64)
static bool ix_moe_decode_kt_served(long kt) {
#define IX_DEC_IS(KT_) if (kt == KT_) return true;
  IX_DEC_KTS(IX_DEC_IS)
#undef IX_DEC_IS
  return false;
}
static bool ix_moe_decode_serves(long Hd, long F) {
  return Hd % 256 == 0 && F % 128 == 0 && ix_moe_decode_kt_served(Hd / 64) && ix_moe_decode_kt_served(F / 64);
}

// Fragment-packed copies of both expert matrices for the decode kernels (each the size of its source).
extern "C" int ix_moe_pack_decode(const void* W1, const void* W2, void* W1f, void* W2f, long E, long Hd, long F,
                                  void* stream) {
  if (!W1 || !W2 || !W1f || !W2f || E <= 0 || Hd <= 0 || F <= 0) return IX_ERR_ARG;
  if (!ix_moe_decode_serves(Hd, F) || !ix_aligned(W1, 16) || !ix_aligned(W2, 16) || !ix_aligned(W1f, 16) ||
      !ix_aligned(W2f, 16))
    return IX_DECLINED;
  const long c1 = E * 2 * F * Hd / 8, c2 = E * Hd * F / 8;
  if ((c1 + 255) / 256 > 0x7fffffffL) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_moe_pack_frag, dim3((unsigned)((c1 + 255) / 256)), dim3(256), 0, st, (const bf16_t*)W1, (bf16_t*)W1f,
                     (int)(2 * F), (int)Hd, (int)(F / 128), 1, c1);
  hipLaunchKernelGGL(k_moe_pack_frag, dim3((unsigned)((c2 + 255) / 256)), dim3(256), 0, st, (const bf16_t*)W2, (bf16_t*)W2f,
                     (int)Hd, (int)F, (int)(Hd / 256), 0, c2);
  return ix_launch_status();
}

// ix_moe_experts for a block map of 32- or 64-row tiles, reading the fragment-packed matrices.
extern "C" int ix_moe_experts_packed(const void* x, long ldx, const int* sorted_token, const float* permuted_prob,
                                     const void* W1f, const void* W2f, const int* tile_meta, long max_tiles, long BM,
                                     void* inter, void* expert_out, long T, long rows, long Hd, long F, void* stream) {
  return ix_moe_experts_packed_footprint(x, ldx, sorted_token, permuted_prob, W1f, W2f, tile_meta, max_tiles, BM, inter,
                                         expert_out, T, rows, Hd, F, 0, stream);
}

extern "C" int ix_moe_experts_packed_footprint(const void* x, long ldx, const int* sorted_token, const float* permuted_prob,
                                               const void* W1f, const void* W2f, const int* tile_meta, long max_tiles, long BM,
                                               void* inter, void* expert_out, long T, long rows, long Hd, long F,
                                               size_t footprint, void* stream) {
  if (!x || !sorted_token || !permuted_prob || !W1f || !W2f || !tile_meta || !inter || !expert_out) return IX_ERR_ARG;
  if (T < 0 || rows < 0 || Hd <= 0 || F <= 0 || max_tiles < 0 || ldx < Hd || (BM != 32 && BM != 64)) return IX_ERR_ARG;
  if (!ix_moe_decode_serves(Hd, F) || (ldx % 8) || !ix_aligned(x, 16) || !ix_aligned(W1f, 16) || !ix_aligned(W2f, 16) ||
      !ix_aligned(inter, 16) || !ix_aligned(expert_out, 16))
    return IX_DECLINED;
  if (rows == 0 || max_tiles == 0) return IX_OK;
  const long nb1 = F / 128, nb2 = Hd / 256;
  const long tiles = max_tiles < rows ? max_tiles : rows;  // every tile has a row
  const long u1 = tiles * nb1 * 4, u2 = tiles * nb2 * 4;
  if (u1 > 0x7ffffff0L || u2 > 0x7ffffff0L) return IX_DECLINED;
  const dim3 g1((unsigned)(8 * ((u1 + 7) / 8))), g2((unsigned)(8 * ((u2 + 7) / 8)));
  const bool once = ix_streams_once((size_t)tiles * 3 * F * Hd * 2, footprint);
  hipStream_t st = (hipStream_t)stream;
#define IX_DEC_FC1_GO(KT_, BM_, ONCE_)                                                                              \
  hipLaunchKernelGGL((k_moe_fc1_dec<KT_, BM_, ONCE_>), g1, dim3(64), 0, st, (const bf16_t*)x, ldx, sorted_token,     \
                     permuted_prob, (const bf16_t*)W1f, tile_meta, (int)max_tiles, (bf16_t*)inter, (int)F, (int)nb1)
#define IX_DEC_FC2_GO(KT_, BM_, ONCE_)                                                                               \
  hipLaunchKernelGGL((k_moe_fc2_dec<KT_, BM_, ONCE_>), g2, dim3(64), 0, st, (const bf16_t*)inter, (const bf16_t*)W2f, \
                     tile_meta, (int)max_tiles, (bf16_t*)expert_out, (int)Hd, (int)F, (int)nb2)
#define IX_DEC_CASE(GO, KT_)                     \
  if (BM == 32 && once) GO(KT_, 32, true);       \
  else if (BM == 32) GO(KT_, 32, false);         \
  else if (once) GO(KT_, 64, true);              \
  else GO(KT_, 64, false);
#define IX_DEC_FC1(KT_) \
  if (Hd / 64 == KT_) { IX_DEC_CASE(IX_DEC_FC1_GO, KT_) }
#define IX_DEC_FC2(KT_) \
  if (F / 64 == KT_) { IX_DEC_CASE(IX_DEC_FC2_GO, KT_) }
  IX_DEC_KTS(IX_DEC_FC1)
  IX_DEC_KTS(IX_DEC_FC2)
#undef IX_DEC_FC1
#undef IX_DEC_FC2
#undef IX_DEC_CASE
#undef IX_DEC_FC1_GO
#undef IX_DEC_FC2_GO
  return ix_launch_status();
}

extern "C" int ix_moe_experts_decode(const void* x, long ldx, const int* sorted_token, const float* permuted_prob,
                                     const void* W1f, const void* W2f, const int* tile_meta, long max_tiles, void* inter,
                                     void* expert_out, long T, long rows, long Hd, long F, void* stream) {
  return ix_moe_experts_packed(x, ldx, sorted_token, permuted_prob, W1f, W2f, tile_meta, max_tiles, 32, inter, expert_out, T,
                               rows, Hd, F, stream);
}

// ---------------------------------------------------------------------------------------------
// A wave sums 512 columns of one token's KC rows (whole 16-byte groups only). The token is uniform in a wave, so its row
// numbers and row addresses are scalar work, and the bf16 form's roundings go through the hardware's pack-convert: it keeps
// a NaN's payload where ix_rbf makes 0x7fc0, but a NaN stays one through the later adds and the store makes it canonical.
// The thread-per-group form below is bound by its own vector instructions instead (a 64-bit division and an integer rounding
// per element and row): 4096 tokens of 8 rows of 2048 columns 41 -> 28 us (5.4 TB/s).
template <int KC, bool FP32>
__global__ __launch_bounds__(256) void k_moe_combine_rows(const bf16_t* __restrict__ expert_out,
                                                          const int* __restrict__ combine_rows, bf16_t* __restrict__ out,
                                                          unsigned waves, unsigned chunks, int Hd) {
  const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (wave >= waves) return;
  const unsigned t = wave / chunks, chunk = wave - t * chunks;
  const int c0 = (int)chunk * 512 + (int)(threadIdx.x & 63) * 8;
  if (c0 >= Hd) return;
  const int* rows = combine_rows + (size_t)t * KC;
  uint4 e[KC];
#pragma unroll
  for (int r = 0; r < KC; ++r) e[r] = *reinterpret_cast<const uint4*>(expert_out + (long)rows[r] * Hd + c0);
  float sum[8];
  ix_unpack8(e[0], sum);
#pragma unroll
  for (int r = 1; r < KC; ++r) {
    float x[8];
    ix_unpack8(e[r], x);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float s0 = sum[i] + x[i], s1 = sum[i + 1] + x[i + 1];
      if constexpr (FP32) {
        sum[i] = s0;
        sum[i + 1] = s1;
      } else {
        ix_rbf2_hw(s0, s1, sum[i], sum[i + 1]);
      }
    }
  }
  uint4 o;
  o.x = ix_pack_bf2_canon_hw(sum[0], sum[1]);
  o.y = ix_pack_bf2_canon_hw(sum[2], sum[3]);
  o.z = ix_pack_bf2_canon_hw(sum[4], sum[5]);
  o.w = ix_pack_bf2_canon_hw(sum[6], sum[7]);
  *reinterpret_cast<uint4*>(out + (size_t)t * Hd + c0) = o;
}

// Any width and alignment, a thread per 8 columns. KC > 0: k known at compile time -- the k row numbers and the k rows are
// requested before the first add, so a thread has k loads in flight instead of one (the sum is the same left-to-right sum).
// KC = 0: any k.
template <int KC>
__global__ __launch_bounds__(256) void k_moe_combine(const bf16_t* __restrict__ expert_out,
                                                     const int* __restrict__ combine_rows,
                                                     bf16_t* __restrict__ out, long T, int Hd, int k, int fp32_acc,
                                                     int vec) {
  const int groups = (Hd + 7) / 8;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= T * groups) return;
  const long t = i / groups;
  const int c0 = (int)(i % groups) * 8;
  float acc[8];
  if constexpr (KC > 0) {
    long row[KC];
    float xv[KC][8];
#pragma unroll
    for (int r = 0; r < KC; ++r) row[r] = combine_rows[t * KC + r];
#pragma unroll
    for (int r = 0; r < KC; ++r) ix_load8(expert_out + row[r] * Hd + c0, Hd - c0, vec != 0, 0.0f, xv[r]);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = xv[0][j];
#pragma unroll
    for (int r = 1; r < KC; ++r) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float sum = acc[j] + xv[r][j];
        acc[j] = fp32_acc ? sum : ix_rbf(sum);
      }
    }
  } else {
    for (int r = 0; r < k; ++r) {
      const long row = combine_rows[t * k + r];
      float xv[8];
      ix_load8(expert_out + row * Hd + c0, Hd - c0, vec != 0, 0.0f, xv);
      if (r == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = xv[j];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float sum = acc[j] + xv[j];
          acc[j] = fp32_acc ? sum : ix_rbf(sum);
        }
      }
    }
  }
  ix_store8_bf16(out + t * Hd + c0, Hd - c0, vec != 0, acc);
}

extern "C" int ix_moe_combine(const void* expert_out, const int* combine_rows, void* out, long T, long Hd, long k,
                              int fp32_acc, void* stream) {
  if (!expert_out || !combine_rows || !out || T < 0 || Hd <= 0 || k <= 0) return IX_ERR_ARG;
  if (T == 0) return IX_OK;
  const long groups = (Hd + 7) / 8;
  const long grid = (T * groups + 255) / 256;
  if (grid > 0x7fffffffL) return IX_DECLINED;
  const int vec = (Hd % 8 == 0) && ix_aligned(expert_out, 16) && ix_aligned(out, 16);
  const long chunks = (Hd + 511) / 512;
  // A wave's 512 columns leave lanes idle in narrow rows, and each row of a token costs the wave its scalar addresses: the fewer
  // the rows, the wider they have to be. us in threads / in waves at 65536 tokens: k = 2 192 columns 14.7 / 15.5, 256 17.6 /
  // 17.6; k = 4 128 17.2 / 19.2, 160 21.7 / 20.4; k = 8 64 18.0 / 28.3, 128 29.3 / 28.4. With fp32 sums, which leave the threads
  // little arithmetic, and more than the caches hold several times over, threads again: 2048 columns, k = 8 469 / 477.
  const long least = k == 2 ? 256 : (k == 4 ? 160 : 128);
  const bool waves = Hd >= least && !(fp32_acc && T * Hd >= (1L << 26)) && T * chunks <= 0x7fffffffL;
  if (vec && waves && (k == 2 || k == 4 || k == 8)) {
#define IX_COMBINE_ROWS(KC_, F_)                                                                                       \
  hipLaunchKernelGGL((k_moe_combine_rows<KC_, F_>), dim3((unsigned)((T * chunks + 3) / 4)), dim3(256), 0,              \
                     (hipStream_t)stream, (const bf16_t*)expert_out, combine_rows, (bf16_t*)out, (unsigned)(T * chunks), \
                     (unsigned)chunks, (int)Hd)
    if (k == 2) { if (fp32_acc) IX_COMBINE_ROWS(2, true); else IX_COMBINE_ROWS(2, false); }
    if (k == 4) { if (fp32_acc) IX_COMBINE_ROWS(4, true); else IX_COMBINE_ROWS(4, false); }
    if (k == 8) { if (fp32_acc) IX_COMBINE_ROWS(8, true); else IX_COMBINE_ROWS(8, false); }
#undef IX_COMBINE_ROWS
    return ix_launch_status();
  }
#define IX_COMBINE(KC_)                                                                                        \
  hipLaunchKernelGGL(k_moe_combine<KC_>, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,             \
                     (const bf16_t*)expert_out, combine_rows, (bf16_t*)out, T, (int)Hd, (int)k, fp32_acc, vec)
  switch (k) {
    case 2: IX_COMBINE(2); break;
    case 4: IX_COMBINE(4); break;
    case 8: IX_COMBINE(8); break;
    default: IX_COMBINE(0); break;
  }
#undef IX_COMBINE
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// The combine with a weight per expert row and any of the eager form's dtypes (moe_batch_invariant.py:276-320 after
// :366-369 `permuted_tokens * permuted_probs.unsqueeze(-1)`): value_r = x[row_r] * w[row_r], summed left to right
// over a token's k rows. The arithmetic dtype is torch's promotion of (token dtype, weight dtype): in bf16 the
// product and every partial sum are rounded to bf16, in fp32 nothing is rounded before the store.
template <typename TIN>
__global__ __launch_bounds__(256) void k_moe_combine_weighted(const TIN* __restrict__ expert_out,
                                                              const float* __restrict__ row_weight,
                                                              const int* __restrict__ combine_rows, void* __restrict__ out,
                                                              long T, int Hd, int k, int arith_bf16, int out_bf16,
                                                              int vec) {
  const int groups = (Hd + 7) / 8;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= T * groups) return;
  const long t = i / groups;
  const int c0 = (int)(i % groups) * 8;
  float acc[8];
  for (int r = 0; r < k; ++r) {
    const long row = combine_rows[t * k + r];
    float xv[8];
    ix_load8(expert_out + row * Hd + c0, Hd - c0, vec != 0, 0.0f, xv);
    if (row_weight) {
      const float w = row_weight[row];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float prod = xv[j] * w;
        xv[j] = arith_bf16 ? ix_rbf(prod) : prod;
      }
    }
    if (r == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = xv[j];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float sum = acc[j] + xv[j];
        acc[j] = arith_bf16 ? ix_rbf(sum) : sum;
      }
    }
  }
  if (out_bf16) {
    ix_store8_bf16((bf16_t*)out + t * Hd + c0, Hd - c0, vec != 0, acc);
  } else {
    float* o = (float*)out + t * Hd + c0;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (c0 + j < Hd) o[j] = acc[j];
  }
}

extern "C" int ix_moe_combine_weighted(const void* expert_out, int in_dtype, const float* row_weight, int arith_dtype,
                                       const int* combine_rows, void* out, int out_dtype, long T, long Hd, long k,
                                       void* stream) {
  if (!expert_out || !combine_rows || !out || T < 0 || Hd <= 0 || k <= 0) return IX_ERR_ARG;
  const auto known = [](int d) { return d == IX_DT_F32 || d == IX_DT_BF16; };
  if (!known(in_dtype) || !known(arith_dtype) || !known(out_dtype)) return IX_DECLINED;
  if (in_dtype == IX_DT_F32 && arith_dtype == IX_DT_BF16) return IX_ERR_ARG;  // promotion never narrows
  if (T == 0) return IX_OK;
  const long groups = (Hd + 7) / 8;
  const long grid = (T * groups + 255) / 256;
  if (grid > 0x7fffffffL) return IX_DECLINED;
  const int vec = (Hd % 8 == 0) && ix_aligned(expert_out, 16) && ix_aligned(out, 16);
  const int ab = arith_dtype == IX_DT_BF16, ob = out_dtype == IX_DT_BF16;
  if (in_dtype == IX_DT_BF16)
    hipLaunchKernelGGL(k_moe_combine_weighted<bf16_t>, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const bf16_t*)expert_out, row_weight, combine_rows, out, T, (int)Hd, (int)k, ab, ob, vec);
  else
    hipLaunchKernelGGL(k_moe_combine_weighted<float>, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const float*)expert_out, row_weight, combine_rows, out, T, (int)Hd, (int)k, ab, ob, vec);
  return ix_launch_status();
}
