// Batch-invariant dense matmuls: the bf16 GEMM behind every linear layer and the LM head, and
// the fp32 GEMM behind the MoE router. Counterpart of the reference's global aten mm/addmm
// override (ops/moe/moe_batch_invariant.py:422-473, ops/mm/mm_tiles.py:127-158) and of its
// pinned non-split-K provider (ops/mm/csrc/cublaslt_pinned.cpp:1-36).
#include "ix_gemm_core.h"
#include "ix_gemm_dense.h"
#include <algorithm>
#include <cmath>

__device__ __forceinline__ void ix_store4(bf16_t* p, int valid, bool vec, const float (&v)[4]) {
  ix_store4_bf16(p, valid, vec, v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void ix_store4(float* p, int valid, bool vec, const float (&v)[4]) {
  if (vec && valid >= 4) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < valid) p[e] = v[e];
  }
}

// Row-max parts a tile writes per row: one, except the four-wave 256 x 256 tile, which writes one per wave column.
template <int BM, int BN, int WM, int WN, int PW>
__host__ __device__ constexpr int ix_gemm_parts_per_tile() {
  return (BM == 256 && BN == 256 && WM == 2 && WN == 2 && PW == 0) ? WN : 1;
}

__device__ __forceinline__ bool ix_tile_of_block(unsigned bid, int nb_m, int nb_n, int* tm, int* tn) {
  return ix_tile_of_run(bid & 7u, bid >> 3, nb_m, nb_n, IX_GEMM_GM, IX_GEMM_GN, tm, tn);
}

// TC = bf16_t: C is the bf16 round of the fp32 accumulator; TC = float: the accumulator itself.
// row_max_parts (optional): [M, parts_ld] fp32, entry (m, tn) = max over the tile's columns of the
// values stored to C (exact, order-free), so a consumer can skip its own max pass over C. part_slots: entries per row, a
// multiple of them per part (the last part takes the rest) where the caller counted another shape's.
template <int BM, int BN, int WM, int WN, typename TC, int PW = 0, bool W_ONCE = false>
__global__ __launch_bounds__((WM * WN + PW) * 64) void k_gemm_bf16_nt(const bf16_t* __restrict__ A, long lda,
                                                              const bf16_t* __restrict__ W, long ldw,
                                                              const bf16_t* __restrict__ bias,
                                                              TC* __restrict__ C, long ldc, int M, int N, int K,
                                                              int nb_m, int nb_n, int vec_store,
                                                              float* __restrict__ row_max_parts, long parts_ld,
                                                              long batch_a, long batch_w, long batch_c, int part_slots) {
  using Cfg = IxGemmCfg<BM, BN, WM, WN, PW, W_ONCE>;
  extern __shared__ __align__(16) char ix_lds[];
  // a batch of independent products (bmm): workgroup row blockIdx.y works on matrices batch strides further on
  A += (long)blockIdx.y * batch_a;
  W += (long)blockIdx.y * batch_w;
  C += (long)blockIdx.y * batch_c;
  int tm, tn;
  if (!ix_tile_of_block(blockIdx.x, nb_m, nb_n, &tm, &tn)) return;
  const long m0 = (long)tm * BM;
  const long n0 = (long)tn * BN;
  const int m_valid = (int)min((long)BM, (long)M - m0);
  const int n_valid = (int)min((long)BN, (long)N - n0);

  // Tile-local buffer descriptors: rows past the matrix fall outside the range and read as 0.
  const ix_rsrc_t x_rsrc = ix_make_rsrc(A + m0 * lda, (uint32_t)(((long)(m_valid - 1) * lda + K) * 2));
  const ix_rsrc_t w_rsrc = ix_make_rsrc(W + n0 * ldw, (uint32_t)(((long)(n_valid - 1) * ldw + K) * 2));
  auto x_row = [&](int r) -> uint32_t { return (r < m_valid) ? (uint32_t)(r * lda * 2) : IX_OOB; };
  auto w_row = [&](int r) -> uint32_t { return (r < n_valid) ? (uint32_t)(r * ldw * 2) : IX_OOB; };

  ix_f32x16 acc[Cfg::MI][Cfg::NI];
  ix_acc_zero<Cfg>(acc);
  ix_gemm_mainloop<Cfg>(x_rsrc, x_row, w_rsrc, w_row, K, ix_lds, acc);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const bool computes = PW == 0 || wave < WM * WN;  // fetching waves hold no results
  float rmax[Cfg::MI];
  // A whole bf16 tile with 16-byte aligned rows takes the wide stores (same values, same places).
  const bool wide = sizeof(TC) == 2 && m_valid == BM && n_valid == BN && (ldc % 8 == 0) && (reinterpret_cast<uintptr_t>(C) % 16 == 0);
  // Compile-time indices throughout: a rolled loop over mi would index the accumulators dynamically and push them to
  // memory. The whole-tile path is instantiated with and without a bias: at 256 values per lane the epilogue is bound by
  // vector-ALU issue, not by the stores (the row maximum costs three instructions per four values and is always taken).
#pragma unroll
  for (int mi = 0; mi < Cfg::MI; ++mi) rmax[mi] = IX_NEG_INF;
  if constexpr (Cfg::MI * Cfg::NI == 16) {
    // the matrix pipeline has drained before the accumulation registers are read by hand below
    asm volatile("s_nop 15\n\ts_nop 15");
  }
  auto whole_tile = [&](auto has_bias_c) {
    constexpr bool HAS_BIAS = decltype(has_bias_c)::value;
    constexpr int NPIECE = Cfg::NI * 2;
    char* buf = ix_lds + wave * ix_store_block32_lds_bytes<NPIECE>();
    ix_static_for<0, Cfg::MI>([&](auto mic) {
      constexpr int mi = decltype(mic)::value;
      uint4 pieces[NPIECE];
      ix_static_for<0, Cfg::NI>([&](auto nic) {
        constexpr int ni = decltype(nic)::value;
        float a16[16];
        ix_acc_read16<(Cfg::MI * Cfg::NI == 16)>(acc[mi][ni], a16);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          uint2 pk[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int q = 2 * p + h;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = a16[q * 4 + e];
            if constexpr (HAS_BIAS) {
              const long n = n0 + wn * Cfg::TN + ni * 32 + ix_acc_row(q * 4, lane);
              const uint2 b4 = *reinterpret_cast<const uint2*>(bias + n);  // n % 4 == 0 and bias is 8-byte aligned
              v[0] = v[0] + __uint_as_float(b4.x << 16);
              v[1] = v[1] + __uint_as_float(b4.x & 0xffff0000u);
              v[2] = v[2] + __uint_as_float(b4.y << 16);
              v[3] = v[3] + __uint_as_float(b4.y & 0xffff0000u);
            }
            rmax[mi] = fmaxf(rmax[mi], fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
            pk[h].x = ix_pack_bf2_hw(v[0], v[1]);
            pk[h].y = ix_pack_bf2_hw(v[2], v[3]);
          }
          pieces[ni * 2 + p] = ix_join_halves(pk[0], pk[1]);
        }
      });
      // whole rows of the wave's TN columns per store instruction instead of 32-byte pieces of 32 rows
      ix_store_block32_via_lds<NPIECE>(buf, pieces,
                                       reinterpret_cast<bf16_t*>(C) + (m0 + wm * Cfg::TM + mi * 32) * ldc + n0 + wn * Cfg::TN,
                                       ldc, 32);
    });
  };
  // Late zero-fills of the ring by other waves' past-the-end fetches must not land on the store buffers.
  if (wide) __syncthreads();
  if (!computes) {
  } else if (wide && (!bias || (reinterpret_cast<uintptr_t>(bias) % 8 == 0))) {
    if (bias) whole_tile(std::true_type{}); else whole_tile(std::false_type{});
  } else {
    ix_static_for<0, Cfg::MI>([&](auto mic) {
      constexpr int mi = decltype(mic)::value;
      const long m = m0 + wm * Cfg::TM + mi * 32 + (lane & 31);
      ix_static_for<0, Cfg::NI>([&](auto nic) {
        constexpr int ni = decltype(nic)::value;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const long n = n0 + wn * Cfg::TN + ni * 32 + ix_acc_row(q * 4, lane);
          const int valid = (int)min(4L, (long)N - n);
          if (valid <= 0 || m >= M) continue;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = acc[mi][ni][q * 4 + e];
            // addmm: the bias joins in fp32 before the single bf16 round.
            if (bias && e < valid) v[e] = v[e] + ix_bf2f(bias[n + e]);
            if (e < valid) rmax[mi] = fmaxf(rmax[mi], v[e]);
          }
          ix_store4(C + m * ldc + n, valid, vec_store != 0, v);
        }
      });
    });
  }
  if (row_max_parts) {
    float* s_max = reinterpret_cast<float*>(ix_lds);  // [WN][BM]
    __syncthreads();                                  // every wave has left the main loop's LDS reads
#pragma unroll
    for (int mi = 0; mi < Cfg::MI; ++mi) {
      float v = fmaxf(rmax[mi], __shfl_xor(rmax[mi], 32, IX_WAVE));
      // rounding is monotonic: the max of the rounded values is the rounded max
      if (sizeof(TC) == 2) v = ix_rbf(v);
      if (computes && lane < 32) s_max[wn * BM + wm * Cfg::TM + mi * 32 + lane] = v;
    }
    __syncthreads();
    // one part per wave column where the streaming form of this tile writes those, without passing through LDS; else one
    constexpr int PPT = ix_gemm_parts_per_tile<BM, BN, WM, WN, PW>();
    const int n_parts = nb_n * PPT, each = part_slots / n_parts;
    for (int r = threadIdx.x; r < m_valid; r += Cfg::NTT) {
#pragma unroll
      for (int p = 0; p < PPT; ++p) {
        float v = s_max[p * BM + r];
        if constexpr (PPT == 1) {
#pragma unroll
          for (int w = 1; w < WN; ++w) v = fmaxf(v, s_max[w * BM + r]);
        }
        const int part = tn * PPT + p, end = part + 1 == n_parts ? part_slots : (part + 1) * each;
        for (int d = part * each; d < end; ++d) row_max_parts[(m0 + r) * parts_ld + d] = v;
      }
    }
  }
}

template <bool ONCE>
using IxStreamSquare = IxGemmCfg<256, 256, 2, 2, 0, ONCE>;
static bool ix_gemm_stream_fits(const void* C, long ldc, long M, long N, long K, const void* bias, long batch) {
  return !bias && batch == 1 && (K % IX_BK == 0) && K / IX_BK >= IX_STREAM_MIN_KT && (N % 8 == 0) && (ldc % 8 == 0) &&
         ix_aligned(C, 16) && ldc * 512 < 0x40000000L;
}

template <int BM, int BN, int WM, int WN, typename TC, int PW = 0, bool W_ONCE = false>
static int ix_gemm_bf16_launch(const bf16_t* A, long lda, const bf16_t* W, long ldw, const bf16_t* bias, TC* C,
                               long ldc, long M, long N, long K, float* parts, long parts_ld, hipStream_t st,
                               long batch = 1, long batch_a = 0, long batch_w = 0, long batch_c = 0, long part_slots = 0) {
  using Cfg = IxGemmCfg<BM, BN, WM, WN, PW>;
  const long nb_m = (M + BM - 1) / BM, nb_n = (N + BN - 1) / BN;
  const long grid = 8 * ((nb_m * nb_n + 7) / 8);  // 8 XCD runs of the tile order, the longest one sets the count
  if (grid > 0x7fffffffL) return IX_DECLINED;
  if (part_slots == 0) part_slots = nb_n * ix_gemm_parts_per_tile<BM, BN, WM, WN, PW>();
  if (parts && parts_ld < part_slots) return IX_ERR_ARG;
  auto kern = k_gemm_bf16_nt<BM, BN, WM, WN, TC, PW, W_ONCE>;
  static bool attr_set = false;  // per instantiation
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES) !=
        hipSuccess)
      return IX_ERR_LAUNCH;
    attr_set = true;
  }
  const int vec = (ldc % 4 == 0) && ix_aligned(C, 4 * sizeof(TC));
  if (batch > 65535) return IX_DECLINED;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid, (unsigned)batch), dim3(Cfg::NTT), Cfg::LDS_BYTES, st, A, lda, W, ldw,
                     bias, C, ldc, (int)M, (int)N, (int)K, (int)nb_m, (int)nb_n, vec, parts, parts_ld, batch_a, batch_w,
                     batch_c, (int)part_slots);
  return ix_launch_status();
}

// Which tile shape runs (0 = choose). Never changes a bit. The choice minimises a cost model: a CU works through
// ceil(tiles / 256) tiles -- the two small shapes two at a time -- at `fixed` us plus K/64 k-tiles each, and no shape streams
// the operands faster than `stream` bytes per us. The figures are a fit to 139 measured shapes (weights 2048 x 4096, 5120 x
// 2048, 12352 x 2048, 8192 x 8192, 151936 x 2048 and x 4096, 1 to 4000 rows) for the five shapes of whole tiles, and to 190
// of the same weights (16 to 7300 rows) for the bands (`bands`: the call is one they serve), whose k-tile costs what the L2
// takes for its operands: 256 CUs pull 10 to 13 TB/s whatever the height. us, without -> with bands: 151936 x 4096 at 192
// rows 290 -> 262, 257 456 -> 358, 320 469 -> 375, 384 492 -> 434, 513 675 -> 587, 769 927 -> 828; 151936 x 2048 at 513 351 ->
// 307; 12352 x 2048 at 320 32 -> 26; 5120 x 2048 at 3090 86 -> 58. One turn of fewer bands than CUs: a CU takes its operands at
// 35 to 39 GB/s where they come from memory, whatever the height (100 rows of 28672 x 4096, 112 column tiles: 64 us
// in bands, 55 in twice as many 128 x 128 tiles; of 40960 x 2048, 160 column tiles, 42 against 51). Bands of equal cost are
// bound by that or by the stream: the lowest (50304 x 2048 at 128 rows 52 -> 49 us). Over 448 points of nineteen weights (65 to
// 4200 rows, no weight read twice out of the caches) the choice is 1.3 % off the fastest shape in the mean and no more than
// 3 % slower than the choice without bands.
#define IX_TILE_BAND 10  // id IX_TILE_BAND + MI: bands of 32 MI rows
#define IX_BAND_CU_RATE 37e3  // bytes per us that a band takes from memory
static int ix_gemm_tile_for(long M, long N, long K, int tile, bool bands) {
  if (tile != 0) return tile;
  // One 128-wide column of tiles (the router's gating product): 128-row tiles once there are enough of them to fill
  // the chip, the small tile below that (2048 x 2048 x 128: 20.7 -> 8.5 us; equal at 16384 rows).
  const bool halves = M <= 32 || ((M + 31) / 32) * ((N + 31) / 32) <= 256;  // of the small tile, see below
  if (M > 128 && N <= 128) return M >= 16384 ? 2 : (halves ? 9 : 6);
  // us_ktile: a tile with its CU to itself; us_ktile_more: one of several (for id 2 and 6: of a pair that shares the CU)
  struct Shape { int id, bm, bn; double us_ktile, us_ktile_more, fixed, stream; };
  static const Shape shapes[] = {{4, 256, 256, 0.98, 1.4, 4.4, 4.4e6},
                                 {IX_TILE_BAND + 7, 224, 256, 1.10, 1.44, 4.4, 5.2e6}, {IX_TILE_BAND + 6, 192, 256, 0.96, 1.27, 4.4, 5.2e6},
                                 {IX_TILE_BAND + 5, 160, 256, 0.78, 1.06, 4.4, 5.2e6}, {IX_TILE_BAND + 4, 128, 256, 0.62, 0.97, 4.4, 5.2e6},
                                  {5, 128, 256, 0.95, 1.1, 7.0, 4.1e6},
                                 {2, 128, 128, 0.51, 0.95, 5.3, 4.7e6}, {1, 32, 256, 0.38, 0.42, 3.7, 4.4e6},
                                 {6, 64, 32, 0.20, 0.29, 1.3, 3.7e6}};  // preference on ties: larger tiles first
  const double kt = (double)((K + 63) / 64);
  int best = 4;
  double best_cost = 1e300;
  // up to 64 rows the 128 x 128 tile with its weights past the caches is the better one (7 rows of 151936 x 4096: 202 us
  // against a band's 226)
  const bool banded = bands && M > 64 && K % IX_BK == 0 && K / IX_BK >= IX_BAND_MIN_KT && N % 8 == 0;
  for (const Shape& sh : shapes) {
    if (sh.id > IX_TILE_BAND && !banded) continue;
    const double tiles = (double)((M + sh.bm - 1) / sh.bm) * (double)((N + sh.bn - 1) / sh.bn);
    const double turns = std::ceil(tiles / 256.0);
    double cost;
    if (sh.id == 4 || sh.id > IX_TILE_BAND) {  // one workgroup per CU streams its tiles: 3 us between two of them
      cost = sh.fixed + turns * (kt * (turns == 1.0 ? sh.us_ktile : sh.us_ktile_more) + 3.0);
    } else if (sh.id == 2 || sh.id == 6) {
      const double pairs = std::floor(turns / 2.0);
      cost = pairs * (sh.fixed + kt * sh.us_ktile_more) + (turns - 2.0 * pairs) * (sh.fixed + kt * sh.us_ktile);
    } else {
      cost = turns * (sh.fixed + kt * (turns == 1.0 ? sh.us_ktile : sh.us_ktile_more));
    }
    const bool band = sh.id > IX_TILE_BAND;
    const double bytes = (double)(N + M) * (double)K * 2.0;
    cost = std::max(cost, band ? sh.fixed + bytes / std::min(sh.stream, IX_BAND_CU_RATE * tiles) : bytes / sh.stream);
    // a later (smaller) shape must win by a margin, but for a band at the cost of a higher one
    if (cost < best_cost * (band ? 0.99 : 0.97) || (band && best > IX_TILE_BAND && cost <= best_cost)) {
      best_cost = cost;
      best = sh.id;
    }
  }
  // The 64 x 32 tile in halves of 32 rows: for few rows its other half only takes room in the ring, whose bytes under way are
  // what a CU's share of the weight waits for (ten stages of 8 KiB instead of six of 12), and at one turn of tiles the halves
  // are on two CUs. With more turns every weight tile is read twice instead. us 64 x 32 / 32 x 32, weights from memory: 2048 x
  // 4096 at 1 row 12.6 / 10.3, 32 13.4 / 12.2, 64 15.8 / 12.2; 5120 x 2048 at 1 8.9 / 7.7, 32 9.4 / 8.5, 64 (320 halves) 10.4 /
  // 12.4; 12352 x 2048 at 32 17.2 / 15.2, 33 16.8 / 19.6; 4096 x 4096 at 64 16.9 / 13.0, 100 14.8 / 17.4; 128 x 4096 at 2000
  // 11.6 / 10.7, 4096 13.0 / 15.5.
  return best == 6 && halves ? 9 : best;
}

// A few rows of x and weight rows 4 KiB apart: where the 128 x 128 tile is the choice, the 32 x 32 one reads the weight faster. TB/s
// 128 x 128 / 32 x 32 at one row of 151936 x 2048: rows 4096 bytes apart 4.9 / 6.0, 4224 5.7 / 6.0, 8192 6.2 / 6.1; K = 1984 in rows of
// 4096 bytes 4.9 / 6.0, without a gap 5.7 / 6.1. Why that distance costs the larger tile is not known, and weights of other sizes
// do not show it, so the rule keeps to what was measured to gain. us at 1 / 8 / 16 rows, 128 x 128 then 32 x 32, K = 2048: 80000 72 72
// 71 - 59 61 65; 100000 76 76 77 - 70 73 78 (on another card 94 93 95 - 75 77 82); 128256 113 108 113 - 92 94 100; 151936 128 128 125 -
// 104 108 117; 200000 143 145 148 - 132 137 150; not 65536 (from card to card 51 to 61 - 53 to 59) nor 250000 (154 157 163 - 161 168
// 184). Less of such rows: K = 1536 of 151936 96 96 94 - 80 86 94, 1024 67 67 68 - 60 66 72. With the row maximum, the norm and the
// logprobs around it 140 140 138 - 119 125 134. With a bias it does not gain (138 139 139 - 136 139 144; 100000 80 80 81 - 89 92 95).
static bool ix_gemm_rows_4k_apart(long M, long N, long K, long ldw) {
  return ldw * 2 == 4096 && K >= 1536 && N >= 80000 && N <= 200000 && M <= (N <= 160000 ? 16 : 8);
}

// Row-max parts per row of C: one per column tile of the shape that runs.
extern "C" long ix_gemm_bf16_n_tiles(long M, long N, long K, int tile) {
  int t = ix_gemm_tile_for(M, N, K, tile, true);
  if (tile == 0 && t == 2 && ix_gemm_rows_4k_apart(M, N, K, K)) t = 9;  // weight rows without a gap
  const long bn = (t == 2) ? 128 : (t == 6 || t == 9) ? 32 : 256;  // ids 1, 3, 4, 5, 7, 8 are 256 wide
  // the four-wave tiles write one part per wave column
  const long per_tile = t > IX_TILE_BAND ? 4 : ((t == 4 || t == 7 || t == 8) ? 2 : 1);
  return N <= 0 ? 0 : per_tile * ((N + bn - 1) / bn);
}

template <typename TC>
static int ix_gemm_bf16_dispatch(const bf16_t* a, long lda, const bf16_t* w, long ldw, const bf16_t* b, TC* c,
                                 long ldc, long M, long N, long K, int tile, float* parts, long parts_ld,
                                 hipStream_t st, long batch = 1, long sa = 0, long sw = 0, long sc = 0) {
  // `tile` only picks which workgroup owns an element (0 = by M); the bits do not depend on it.
#define IX_BATCH_ARGS , batch, sa, sw, sc, slots
  const bool bands_fit = sizeof(TC) == 2 && ix_gemm_stream_fits(c, ldc, M, N, K, b, batch) && K / IX_BK >= IX_BAND_MIN_KT;
  // with row-max parts the choice has to be the one ix_gemm_bf16_n_tiles made from the sizes alone
  const long rows = M * (batch > 1 ? batch : 1);
  int id = ix_gemm_tile_for(rows, N, K, tile, parts || bands_fit);
  long slots = 0;
  if (id > IX_TILE_BAND && !bands_fit) {
    if (tile != 0) return IX_DECLINED;
    // Chosen by size for a call with a bias, an fp32 result or unaligned rows: the shape that the model takes without bands
    // fills a band's four slots per tile. The tiles of 32 columns have more parts than that: the 128 x 128 one in their place.
    // us in the 256-row tile / here, with a bias: 128 rows of 151936 x 2048 277 / 154, 385 of 12352 x 2048 76 / 39, 300 of
    // 40000 x 768 69 / 44; with an fp32 result 214 / 172, 54 / 37, 65 / 41.
    id = ix_gemm_tile_for(rows, N, K, 0, false);
    if (id == 6 || id == 9) id = 2;
    slots = 4 * ((N + 255) / 256);
  }
  if (tile == 0 && id == 2 && batch == 1) {
    if (!b && ix_gemm_rows_4k_apart(M, N, K, ldw) && (!parts || K == ldw)) id = 9;
    else if (parts && ix_gemm_rows_4k_apart(M, N, K, K)) slots = (N + 31) / 32;  // counted for a product without these
  }
  switch (id) {
    case 1: return ix_gemm_bf16_launch<32, 256, 1, 4, TC, 4>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 2:
      if (batch == 1 && ix_gemm_once((M + 127) / 128, N, K))
        return ix_gemm_bf16_launch<128, 128, 2, 2, TC, 0, true>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
      return ix_gemm_bf16_launch<128, 128, 2, 2, TC>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 3: return ix_gemm_bf16_launch<256, 256, 2, 4, TC>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 4:
      if constexpr (sizeof(TC) == 2) {
        // with one tile per workgroup too (12352 x 2048 at 700 rows 53 -> 42 us, 8192 x 8192 at 1100 157 -> 145)
        if (ix_gemm_stream_fits(c, ldc, M, N, K, b, batch))
          return ix_gemm_bf16_stream_launch<IxStreamSquare>(a, lda, w, ldw, (bf16_t*)c, ldc, M, N, K, parts, parts_ld, st);
      }
      [[fallthrough]];
    case 7:  // the same tile, one tile per workgroup
      return ix_gemm_bf16_launch<256, 256, 2, 2, TC>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 5: return ix_gemm_bf16_launch<128, 256, 2, 4, TC>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 6: return ix_gemm_bf16_launch<64, 32, 2, 1, TC, 2>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 9: return ix_gemm_bf16_launch<32, 32, 1, 1, TC, 2>(a, lda, w, ldw, b, c, ldc, M, N, K, parts, parts_ld, st IX_BATCH_ARGS);
    case 8:  // the streaming form whatever the number of tiles (declines what it does not serve)
      if constexpr (sizeof(TC) == 2) {
        if (ix_gemm_stream_fits(c, ldc, M, N, K, b, batch))
          return ix_gemm_bf16_stream_launch<IxStreamSquare>(a, lda, w, ldw, (bf16_t*)c, ldc, M, N, K, parts, parts_ld, st);
      }
      return IX_DECLINED;
    case IX_TILE_BAND + 4:  // bands of 128, 160, 192, 224 rows (decline what the streaming form does not serve)
    case IX_TILE_BAND + 5:
    case IX_TILE_BAND + 6:
    case IX_TILE_BAND + 7:
      if constexpr (sizeof(TC) == 2) {
        if (bands_fit) return ix_gemm_bf16_bands_launch(id - IX_TILE_BAND, a, lda, w, ldw, (bf16_t*)c, ldc, M, N, K, parts, parts_ld, st);
      }
      return IX_DECLINED;
    default: return IX_ERR_ARG;
  }
#undef IX_BATCH_ARGS
}

extern "C" int ix_gemm_bf16_nt(const void* A, long lda, const void* W, long ldw, const void* bias, void* C,
                               int c_dtype, long ldc, long M, long N, long K, int tile, float* row_max_parts,
                               long parts_ld, void* stream) {
  if (!A || !W || !C || M < 0 || N <= 0 || K <= 0) return IX_ERR_ARG;
  if (lda < K || ldw < K || ldc < N) return IX_ERR_ARG;
  if (c_dtype != IX_DT_BF16 && c_dtype != IX_DT_F32) return IX_DECLINED;
  // 16-byte row chunks: every row start and K itself must be a multiple of 8 elements.
  if ((K % 8) || (lda % 8) || (ldw % 8) || !ix_aligned(A, 16) || !ix_aligned(W, 16)) return IX_DECLINED;
  if (M > 0x7fffffffL || N > 0x7fffffffL || K > 0x7fffffffL) return IX_DECLINED;
  if (lda * 2 * 256 >= 0x40000000L || ldw * 2 * 256 >= 0x40000000L) return IX_DECLINED;  // tile offsets < 1 GiB
  if (M == 0) return IX_OK;
  hipStream_t st = (hipStream_t)stream;
  const bf16_t *a = (const bf16_t*)A, *w = (const bf16_t*)W, *b = (const bf16_t*)bias;
  if (c_dtype == IX_DT_BF16)
    return ix_gemm_bf16_dispatch(a, lda, w, ldw, b, (bf16_t*)C, ldc, M, N, K, tile, row_max_parts, parts_ld, st);
  return ix_gemm_bf16_dispatch(a, lda, w, ldw, b, (float*)C, ldc, M, N, K, tile, row_max_parts, parts_ld, st);
}

// aten::bmm of the override (ops/moe/moe_batch_invariant.py:453-464): `batch` independent products in ONE launch, each
// exactly the product ix_gemm_bf16_nt computes (same tiles, same K order, same bits); matrix b of an operand starts
// b * stride elements after matrix 0. The tile shape is chosen for the whole batch (rows M * batch).
extern "C" int ix_gemm_bf16_nt_batched(const void* A, long lda, long stride_a, const void* W, long ldw, long stride_w,
                                       void* C, long ldc, long stride_c, long batch, long M, long N, long K, int tile,
                                       void* stream) {
  if (!A || !W || !C || batch < 0 || M < 0 || N <= 0 || K <= 0) return IX_ERR_ARG;
  if (lda < K || ldw < K || ldc < N) return IX_ERR_ARG;
  if ((K % 8) || (lda % 8) || (ldw % 8) || (stride_a % 8) || (stride_w % 8) || !ix_aligned(A, 16) || !ix_aligned(W, 16))
    return IX_DECLINED;
  if (M > 0x7fffffffL || N > 0x7fffffffL || K > 0x7fffffffL) return IX_DECLINED;
  if (lda * 2 * 256 >= 0x40000000L || ldw * 2 * 256 >= 0x40000000L) return IX_DECLINED;
  if (M == 0 || batch == 0) return IX_OK;
  return ix_gemm_bf16_dispatch((const bf16_t*)A, lda, (const bf16_t*)W, ldw, (const bf16_t*)nullptr, (bf16_t*)C, ldc, M,
                               N, K, tile, (float*)nullptr, 0, (hipStream_t)stream, batch, stride_a, stride_w, stride_c);
}

// ---------------------------------------------------------------------------------------------
// fp32 GEMM (router gating): C[m, n] = sum_k A[m, k] * W[n, k], A bf16 (widened exactly) or
// fp32, W fp32, C fp32. One instruction, v_mfma_f32_32x32x2_f32; instruction j consumes
// k = 2j (lane group 0) and 2j+1 (lane group 1); instructions accumulate left to right.
#define IX_F32_BM 64
#define IX_F32_BN 128
#define IX_F32_BK 32
#define IX_F32_PITCH 33

template <typename TA>
__global__ __launch_bounds__(256) void k_gemm_f32_nt(const TA* __restrict__ A, long lda,
                                                     const float* __restrict__ W, long ldw,
                                                     float* __restrict__ C, long ldc, int M, int N, int K) {
  __shared__ float sA[IX_F32_BM * IX_F32_PITCH];
  __shared__ float sW[IX_F32_BN * IX_F32_PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;  // 2 x 2 waves, wave tile 32 x 64
  const long m0 = (long)blockIdx.x * IX_F32_BM;
  const long n0 = (long)blockIdx.y * IX_F32_BN;
  ix_f32x16 acc[2];
#pragma unroll
  for (int ni = 0; ni < 2; ++ni)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[ni][i] = 0.0f;

  for (int k0 = 0; k0 < K; k0 += IX_F32_BK) {
    // stage A: 64 rows x 32 k, W: 128 rows x 32 k; one element per thread per pass
    for (int q = tid; q < IX_F32_BM * IX_F32_BK; q += 256) {
      const int r = q >> 5, c = q & 31;
      const long m = m0 + r;
      float v = 0.0f;
      if (m < M && k0 + c < K) {
        if constexpr (sizeof(TA) == 2) v = ix_bf2f(A[m * lda + k0 + c]);
        else v = A[m * lda + k0 + c];
      }
      sA[r * IX_F32_PITCH + c] = v;
    }
    for (int q = tid; q < IX_F32_BN * IX_F32_BK; q += 256) {
      const int r = q >> 5, c = q & 31;
      const long n = n0 + r;
      sW[r * IX_F32_PITCH + c] = (n < N && k0 + c < K) ? W[n * ldw + k0 + c] : 0.0f;
    }
    __syncthreads();
    const int fr = lane & 31, fg = lane >> 5;
#pragma unroll
    for (int j = 0; j < IX_F32_BK / 2; ++j) {
      const float a = sA[(wm * 32 + fr) * IX_F32_PITCH + 2 * j + fg];
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const float b = sW[(wn * 64 + ni * 32 + fr) * IX_F32_PITCH + 2 * j + fg];
        acc[ni] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[ni], 0, 0, 0);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int ni = 0; ni < 2; ++ni) {
    const long n = n0 + wn * 64 + ni * 32 + (lane & 31);
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const long m = m0 + wm * 32 + ix_acc_row(i, lane);
      if (m < M) C[m * ldc + n] = acc[ni][i];
    }
  }
}

extern "C" int ix_gemm_f32_nt(const void* A, int a_dtype, long lda, const void* W, long ldw, void* C, long ldc,
                              long M, long N, long K, void* stream) {
  if (!A || !W || !C || M < 0 || N <= 0 || K <= 0) return IX_ERR_ARG;
  if (lda < K || ldw < K || ldc < N) return IX_ERR_ARG;
  if (a_dtype != IX_DT_F32 && a_dtype != IX_DT_BF16) return IX_DECLINED;
  if (M > 0x7fffffffL || N > 0x7fffffffL || K > 0x7fffffffL) return IX_DECLINED;
  if (M == 0) return IX_OK;
  const long gm = (M + IX_F32_BM - 1) / IX_F32_BM, gn = (N + IX_F32_BN - 1) / IX_F32_BN;
  if (gn > 65535) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  if (a_dtype == IX_DT_BF16)
    hipLaunchKernelGGL((k_gemm_f32_nt<bf16_t>), dim3((unsigned)gm, (unsigned)gn), dim3(256), 0, st,
                       (const bf16_t*)A, lda, (const float*)W, ldw, (float*)C, ldc, (int)M, (int)N, (int)K);
  else
    hipLaunchKernelGGL((k_gemm_f32_nt<float>), dim3((unsigned)gm, (unsigned)gn), dim3(256), 0, st,
                       (const float*)A, lda, (const float*)W, ldw, (float*)C, ldc, (int)M, (int)N, (int)K);
  return ix_launch_status();
}
