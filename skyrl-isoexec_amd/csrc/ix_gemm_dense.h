// Dense streaming products: the tile order, the tile sequence, the kernel and its launch, for the 256 x 256 tile (pipeline F,
// ix_gemm.hip) and for bands of 32 MI rows (pipeline G, ix_gemm_bands.hip: a file of its own, the code is long to compile).
#pragma once
#include "ix_gemm_bands.h"
#include "../../include/isoexec_hip.h"

// Workgroup -> tile map. Hardware hands consecutive workgroup ids to the 8 XCDs round-robin, and each XCD has
// its own L2. The tiles are put in one order -- groups of GM M-tiles x GN weight tiles, about what an XCD's 32
// CUs hold at a time, so that a group pulls GM activation tiles and GN weight tiles through the L2 for GM * GN
// tiles; groups run down the M-tiles of GN weight-tile columns before moving to the next columns -- and that
// order is cut into 8 equal runs, one per XCD: every XCD gets the same number of tiles whatever the shape, and
// a weight tile is fetched by one L2 (two where a run ends inside its column group).
#ifndef IX_GEMM_GM
#define IX_GEMM_GM 8  // M-tiles of a group
#endif
#ifndef IX_GEMM_GN
#define IX_GEMM_GN 4  // weight tiles of a group
#endif
// Tile number idx of XCD xcd's run of that order, for groups of GM x GN tiles.
__device__ __forceinline__ bool ix_tile_of_run(unsigned xcd, unsigned idx, int nb_m, int nb_n, int GM, int GN, int* tm,
                                               int* tn) {
  // 32-bit arithmetic throughout (the launch refuses more than 2^31 tiles): a 64-bit division costs a workgroup
  // about a microsecond before its first fetch.
  const unsigned tiles = (unsigned)nb_m * (unsigned)nb_n;
  // this XCD's run of the tile order: [tiles * xcd / 8, tiles * (xcd + 1) / 8)
  const unsigned q = tiles >> 3, r = tiles & 7u;
  const unsigned lo = q * xcd + ((r * xcd) >> 3), hi = q * (xcd + 1) + ((r * (xcd + 1)) >> 3);
  const unsigned l = lo + idx;
  if (l >= hi) return false;
  const unsigned per_ngroup = (unsigned)GN * (unsigned)nb_m;
  const unsigned ng = l / per_ngroup;
  const unsigned rem = l - ng * per_ngroup;
  const int gn = min(GN, nb_n - (int)ng * GN);  // width of this (possibly last) column group
  const unsigned per_mgroup = (unsigned)GM * (unsigned)gn;
  const unsigned mg = rem / per_mgroup;
  const unsigned r2 = rem - mg * per_mgroup;
  const int gm = min(GM, nb_m - (int)mg * GM);
  const unsigned nl = r2 / (unsigned)gm, ml = r2 - nl * (unsigned)gm;
  *tm = (int)mg * GM + (int)ml;
  *tn = (int)ng * GN + (int)nl;
  return true;
}

// ---- the streaming form of the four-wave 256 x 256 tile (pipeline F) -----------------------------------------------
// bf16 output without bias, K a multiple of 64 with at least IX_STREAM_MIN_KT k-tiles, N a multiple of 8, rows of C
// 16-byte aligned. A workgroup takes every (gridDim.x / 8)-th tile of its XCD's run of the tile order.
// Tile sequence of the dense product: position idx of XCD xcd's run of the tile order above; Cfg::BM rows a tile, Cfg::WN
// row-max parts a tile and row.
template <typename Cfg>
struct IxDenseStreamSeq {
  const bf16_t* A;
  const bf16_t* W;
  bf16_t* C;
  float* parts;
  long lda, ldw, ldc, parts_ld;
  int M, N, K, nb_m, nb_n, gm, gn;
  __device__ __forceinline__ bool locate(unsigned xcd, unsigned idx, IxStreamTile& t) const {
    int tm, tn;
    if (!ix_tile_of_run(xcd, idx, nb_m, nb_n, gm, gn, &tm, &tn)) return false;
    const long m0 = (long)tm * Cfg::BM, n0 = (long)tn * 256;
    t.x = A + m0 * lda;
    t.w = W + n0 * ldw;
    t.c = C + m0 * ldc + n0;
    t.part = parts ? parts + m0 * parts_ld + tn * Cfg::WN : nullptr;
    t.mv = (int)min((long)Cfg::BM, (long)M - m0);
    t.nv = (int)min(256L, (long)N - n0);
    return true;
  }
};

// Cfg: the 256 x 256 tile (pipeline F) or a band of 32 MI rows (pipeline G).
template <typename Cfg, bool PARTS>
__global__ __launch_bounds__(256) void k_gemm_bf16_nt_stream(const bf16_t* __restrict__ A, long lda,
                                                             const bf16_t* __restrict__ W, long ldw,
                                                             bf16_t* __restrict__ C, long ldc, int M, int N, int K,
                                                             int nb_m, int nb_n, int gm, int gn,
                                                             float* __restrict__ row_max_parts, long parts_ld) {
  extern __shared__ __align__(16) char ix_lds[];
  IxPlainStreamJob<Cfg, IxDenseStreamSeq<Cfg>, PARTS> job;
  job.seq.gm = gm;
  job.seq.gn = gn;
  job.seq.A = A;
  job.seq.lda = lda;
  job.seq.W = W;
  job.seq.ldw = ldw;
  job.seq.C = C;
  job.seq.ldc = ldc;
  job.seq.M = M;
  job.seq.N = N;
  job.seq.K = K;
  job.seq.nb_m = nb_m;
  job.seq.nb_n = nb_n;
  job.seq.parts = row_max_parts;
  job.seq.parts_ld = parts_ld;
  if constexpr (Cfg::WM == 2) ix_gemm_stream4<Cfg>(job, K / IX_BK, ix_lds);
  else ix_gemm_bands<Cfg>(job, K / IX_BK, ix_lds);
}

// Weights with one reader in the launch (ix_dma16): a single row tile, and more of them than the caches would keep for the
// next launch anyway.
static bool ix_gemm_once(long nb_m, long N, long K) { return nb_m == 1 && N * K * 2 >= (64L << 20); }

template <auto KERN, typename... Args>
static int ix_gemm_stream_start(int lds, hipStream_t st, Args... args) {
  static bool attr_set = false;  // per kernel
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return IX_ERR_LAUNCH;
    attr_set = true;
  }
  hipLaunchKernelGGL(KERN, dim3(IX_STREAM_WORKGROUPS), dim3(256), lds, st, args...);
  return ix_launch_status();
}

// CFG<once>: the tile (a product without parts takes the same kernel in the bands: an empty descriptor drops its stores)
template <template <bool> class CFG>
static int ix_gemm_bf16_stream_launch(const bf16_t* A, long lda, const bf16_t* W, long ldw, bf16_t* C, long ldc, long M,
                                      long N, long K, float* parts, long parts_ld, hipStream_t st) {
  using Cfg = CFG<false>;
  const long nb_m = (M + Cfg::BM - 1) / Cfg::BM, nb_n = (N + 255) / 256;
  if (nb_m * nb_n > 0x7fffffffL) return IX_DECLINED;
  if (parts && parts_ld < nb_n * Cfg::WN) return IX_ERR_ARG;
  // Group shape of the tile order: with many row tiles the activations are the operand that streams, and a group
  // that is wider in weight tiles re-uses each activation tile more often (163840 x 2048 x 12352: 6.40 -> 6.20 ms,
  // 32768 x 2048 x 151936: 15.7 -> 15.5); with few row tiles the default serves the weights better.
  const int gm = nb_m >= 64 ? 4 : IX_GEMM_GM, gn = nb_m >= 64 ? 16 : IX_GEMM_GN;
#define IX_STREAM_GO(PARTS_, ONCE_)                                                                                       \
  return ix_gemm_stream_start<k_gemm_bf16_nt_stream<CFG<ONCE_>, PARTS_>>(Cfg::LDS_BYTES, st, A, lda, W, ldw, C, ldc, (int)M, \
                                                                         (int)N, (int)K, (int)nb_m, (int)nb_n, gm, gn, parts, parts_ld)
  if (ix_gemm_once(nb_m, N, K)) {
    if (parts || Cfg::WM == 1) IX_STREAM_GO(true, true);
    if constexpr (Cfg::WM == 2) IX_STREAM_GO(false, true);
  }
  if (parts || Cfg::WM == 1) IX_STREAM_GO(true, false);
  if constexpr (Cfg::WM == 2) IX_STREAM_GO(false, false);
  return IX_ERR_ARG;
#undef IX_STREAM_GO
}

// ix_gemm_bands.hip: bands of 128, 160, 192 or 224 rows
int ix_gemm_bf16_bands_launch(int mi, const bf16_t* A, long lda, const bf16_t* W, long ldw, bf16_t* C, long ldc, long M, long N,
                              long K, float* parts, long parts_ld, hipStream_t st);
