// Streaming forms of the expert GEMMs that several files compile: the tile order, the second GEMM (256 x 256 tiles in
// ix_moe.hip, bands of 32 MI rows here) and the first GEMM in bands, with their launch (ix_moe_bands_*.hip).
#pragma once
#include "ix_gemm_bands.h"
#include "../../include/isoexec_hip.h"

// Workgroup -> tile: hardware hands consecutive workgroup ids to the 8 XCDs round-robin and each XCD has its own
// L2, so the tile order (row tile major, column tile minor: an expert's tiles are adjacent) is cut into 8 equal
// runs, one per XCD. The ~32 tiles an XCD works on at a time then belong to one or two experts: an expert's
// weights and a row tile's activations go through one L2 once, instead of through all eight.
__device__ __forceinline__ bool ix_moe_tile_of_block(unsigned bid, int n_row_tiles, int nb_n, int* mt, int* nt) {
  const unsigned xcd = bid & 7u;
  const unsigned idx = bid >> 3;
  const unsigned tiles = (unsigned)n_row_tiles * (unsigned)nb_n;  // < 2^31: the launch checks the bound
  const unsigned q = tiles >> 3, r = tiles & 7u;
  const unsigned lo = q * xcd + ((r * xcd) >> 3), hi = q * (xcd + 1) + ((r * (xcd + 1)) >> 3);
  const unsigned l = lo + idx;
  if (l >= hi) return false;
  *mt = (int)(l / (unsigned)nb_n);
  *nt = (int)(l - (unsigned)*mt * (unsigned)nb_n);
  return true;
}

// ---- streaming form of the second expert GEMM (pipeline F): the four-wave 256 x 256 tile, Hd a multiple of 256, F a
// multiple of 64 with at least IX_STREAM_MIN_KT k-tiles. A workgroup takes every (gridDim.x / 8)-th tile of its XCD's run
// of the (row tile, column tile) order of ix_moe_tile_of_block.
struct IxMoeFc2Seq {
  const bf16_t* inter;
  const bf16_t* W2;
  bf16_t* out;
  const int* meta;
  int max_tiles, Hd, nb_n, K;  // K = F
  long lda, ldw, ldc, parts_ld;  // F, F, Hd, unused
  __device__ __forceinline__ bool locate(unsigned xcd, unsigned idx, IxStreamTile& t) const {
    int mt, nt;
    if (!ix_moe_tile_of_block(xcd + 8u * idx, meta[0], nb_n, &mt, &nt)) return false;
    const long e = meta[1 + mt], row0 = meta[1 + max_tiles + mt];
    t.x = inter + row0 * K;
    t.w = W2 + (e * Hd + (long)nt * 256) * K;
    t.c = out + row0 * Hd + (long)nt * 256;
    t.part = nullptr;
    t.mv = meta[1 + 2 * max_tiles + mt];
    t.nv = 256;
    return true;
  }
};

// Cfg: the 256 x 256 tile (pipeline F) or a band of 32 MI rows (pipeline G).
template <typename Cfg>
__global__ __launch_bounds__(256) void k_moe_fc2_stream(const bf16_t* __restrict__ inter, const bf16_t* __restrict__ W2,
                                                        const int* __restrict__ meta, int max_tiles,
                                                        bf16_t* __restrict__ out, int Hd, int F, int nb_n) {
  extern __shared__ __align__(16) char ix_lds[];
  IxPlainStreamJob<Cfg, IxMoeFc2Seq, false> job;
  job.seq.inter = inter;
  job.seq.W2 = W2;
  job.seq.out = out;
  job.seq.meta = meta;
  job.seq.max_tiles = max_tiles;
  job.seq.Hd = Hd;
  job.seq.nb_n = nb_n;
  job.seq.K = F;
  job.seq.lda = F;
  job.seq.ldw = F;
  job.seq.ldc = Hd;
  job.seq.parts_ld = 0;
  if constexpr (Cfg::WM == 2) ix_gemm_stream4<Cfg>(job, F / IX_BK, ix_lds);
  else ix_gemm_bands<Cfg>(job, F / IX_BK, ix_lds);
}

// ---- the first expert GEMM in bands of 32 MI rows (pipeline G) --------------------------------------------------------
// IxMoeFc1StreamJob for one row of waves: a wave holds 32 gate columns and their 32 up columns (two blocks), so a lane ends
// with 16 consecutive output columns of its token (row rho = 8 g + 4 h + i of either block is column 16 h + 4 g + i of the
// wave's 32); one exchange between neighbouring lanes leaves a pair with 32 contiguous bytes of one token. The chains of
// block mi are micro-steps 64 mi .. 64 mi + 63 (the first eight k-tiles), the exchange and the two stores 16 steps of the
// two k-tiles after them. Same operations in the same order per element.
template <typename Cfg>
struct IxMoeFc1BandJob {
  static constexpr int MI = Cfg::MI, NCH = 64 * MI, NSK = 10;
  static constexpr int DMA_IDLE = 3;  // short of scalar registers (ix_dma16)
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
  ix_rsrc_t nx_xr, nx_wr;
  bool has_next;
  int nx_row0, c_row0, nx_nrows, nx_n0h, c_nrows, c_n0h;
  uint32_t xvo[MI];             // this thread's activation chunks (gathered token rows)
  uint32_t wv;                  // its next weight chunk
  int w_stU, w_stN, w_st0;      // gate -> up rows, to the next wave's gate rows, back to chunk 0 (bytes)
  float prob[MI];               // routing weights of this lane's tokens
  ix_rsrc_t p_ir;               // pending tile: descriptor of its part of inter
  uint32_t p_voff;
  uint32_t pg[MI][8], pu[MI][8];  // pending gate / up values, two bf16 per register; pg takes the chain's result
  uint32_t ta[2][4];
  float g0, g1, a0, a1;           // a chain in flight
  uint32_t g_tok[MI], g_prob[MI];

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
    nx_wr = ix_make_rsrc(W1 + (e * 2 * F + nx_n0h) * Hd, (uint32_t)(((long)F + 128) * Hd * 2));
  }
  __device__ __forceinline__ uint32_t kb() const {
    return (uint32_t)(((threadIdx.x & 7) ^ ix_swz8(threadIdx.x >> 3)) * 16);  // rows 32 apart share the swizzle
  }
  __device__ __forceinline__ uint32_t row_off(int j, uint32_t tok) const {  // a row the tile does not have: out of range
    return ((int)(threadIdx.x >> 3) + 32 * j < nx_nrows) ? tok * (uint32_t)(ldx * 2) + kb() : IX_OOB;
  }
  __device__ __forceinline__ void take_gathers() {
    ix_static_for<0, MI>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      xvo[j] = row_off(j, ix_landed(g_tok[j]));
    });
    ix_static_for<0, MI>([&](auto mc) { prob[decltype(mc)::value] = __uint_as_float(ix_landed(g_prob[decltype(mc)::value])); });
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
    for (int i = 0; i < MI; ++i) {
      prob[i] = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c) pg[i][c] = pu[i][c] = 0u;
    }
    g0 = g1 = a0 = a1 = 0.0f;
    return has_next;
  }
  __device__ __forceinline__ void open_next() {
    idx += stride;
    locate();
    const int last = rows - 1;
    ix_static_for<0, MI>([&](auto jc) {  // token ids of the next tile's rows
      constexpr int j = decltype(jc)::value;
      g_tok[j] = ix_load4_uncounted(sorted_token, (uint32_t)min(nx_row0 + (int)(threadIdx.x >> 3) + 32 * j, last) * 4u);
    });
    ix_static_for<0, MI>([&](auto mc) {  // routing weights of the current tile's
      constexpr int mi = decltype(mc)::value;
      g_prob[mi] = ix_load4_uncounted(permuted_prob, (uint32_t)min(c_row0 + (int)(threadIdx.x & 31) + 32 * mi, last) * 4u);
    });
  }
  __device__ __forceinline__ void first_voffs() {
    const int r0 = threadIdx.x >> 3;
    uint32_t tok[MI];  // nothing is in flight yet: ordinary loads
#pragma unroll
    for (int j = 0; j < MI; ++j) tok[j] = (uint32_t)sorted_token[min(nx_row0 + r0 + 32 * j, rows - 1)];
#pragma unroll
    for (int j = 0; j < MI; ++j) xvo[j] = row_off(j, tok[j]);
    // weight tile row r0 + 32 j: wave j / 2, gate (j even) or up block: weight row [up: F] + 32 (j / 2) + lane_col(r0)
    const int lane_col = 16 * ((r0 >> 2) & 1) + 4 * (r0 >> 3) + (r0 & 3);
    const int row_bytes = Hd * 2;
    wv = (uint32_t)(lane_col * row_bytes) + kb();
    w_stU = __builtin_amdgcn_readfirstlane(F * row_bytes);
    w_stN = __builtin_amdgcn_readfirstlane((32 - F) * row_bytes);
    w_st0 = __builtin_amdgcn_readfirstlane(-(F + 96) * row_bytes);
  }
  template <int J>
  __device__ __forceinline__ uint32_t x_voff() const { return xvo[J]; }
  template <int J>
  __device__ __forceinline__ uint32_t w_voff() {
    const uint32_t v = wv;
    asm volatile("v_add_u32 %0, %1, %0" : "+v"(wv) : "s"(J == 7 ? w_st0 : ((J & 1) ? w_stN : w_stU)));
    return v;
  }
  __device__ __forceinline__ void turn_offsets() { take_gathers(); }
  __device__ __forceinline__ void advance() {
    c_row0 = nx_row0;
    c_nrows = nx_nrows;
    c_n0h = nx_n0h;
  }
  template <typename Acc>
  __device__ __forceinline__ void drain(Acc& acc) {
    ix_static_for<0, MI>([&](auto mc) {
      constexpr int mi = decltype(mc)::value;
      float g16[16], u16[16];
      ix_acc_read16<true>(acc[mi][0], g16);
      ix_acc_read16<true>(acc[mi][1], u16);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        pg[mi][i] = ix_pack_bf2_hw(g16[2 * i], g16[2 * i + 1]);
        pu[mi][i] = ix_pack_bf2_hw(u16[2 * i], u16[2 * i + 1]);
      }
      ix_pin8(pg[mi]);
      ix_pin8(pu[mi]);
    });
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // after the exchange a lane holds piece (lane % 2) of the two tokens of its pair
    const int r = lane & 30, c = wave * 32 + 16 * (lane >> 5) + 8 * (lane & 1);
    p_ir = ix_make_rsrc(inter + (long)c_row0 * F + c_n0h, (uint32_t)(((long)(c_nrows - 1) * F + 128) * 2));
    p_voff = (uint32_t)(((long)r * F + c) * 2);
  }
  static constexpr bool is_store(int i) { return i >= NCH && (i & 15) >= 8 && (i & 15) < 10; }
  static __device__ __forceinline__ int w_frag_row(int ni, int rho) { return ni * 32 + rho; }
  template <int I>
  __device__ __forceinline__ void micro() {
    if constexpr (I < NCH) {
      constexpr int mi = I / 64, c = (I & 63) >> 3, st = I & 7;
      if constexpr (st == 0) {
        g0 = __uint_as_float(pg[mi][c] << 16);
        g1 = __uint_as_float(pg[mi][c] & 0xffff0000u);
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
        const float u0 = __uint_as_float(pu[mi][c] << 16), u1 = __uint_as_float(pu[mi][c] & 0xffff0000u);
        ix_rbf2_hw(a0 * u0, a1 * u1, a0, a1);
      } else {
        pg[mi][c] = ix_pack_bf2_hw(a0 * prob[mi], a1 * prob[mi]);
      }
    } else {
      constexpr int mi = (I - NCH) >> 4, q = (I - NCH) & 15;
      if constexpr (q < 8) {  // piece p, dword d of the lane's 32 bytes: pg[mi][4 p + d]
        constexpr int d = q >> 1, t = q & 1;
        ta[t][d] = ix_quad_exchange<1, t != 0>(pg[mi][d], pg[mi][4 + d]);
      } else if constexpr (q < 10) {
        constexpr int t = q - 8;  // token t of the pair
        ix_buffer_store16<IX_STREAM_STORE_NT_FC1>(make_uint4(ta[t][0], ta[t][1], ta[t][2], ta[t][3]), p_ir,
                          p_voff == IX_OOB ? IX_OOB : p_voff + (uint32_t)((long)(mi * 32 + t) * F * 2));
      }
    }
  }
};

template <typename Cfg>
__global__ __launch_bounds__(256) void k_moe_fc1_glu_bands(const bf16_t* __restrict__ x, long ldx, int T, int rows,
                                                           const int* __restrict__ sorted_token,
                                                           const float* __restrict__ permuted_prob,
                                                           const bf16_t* __restrict__ W1, const int* __restrict__ meta,
                                                           int max_tiles, bf16_t* __restrict__ inter, int Hd, int F,
                                                           int nb_n) {
  extern __shared__ __align__(16) char ix_lds[];
  IxMoeFc1BandJob<Cfg> job;
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
  ix_gemm_bands<Cfg>(job, Hd / IX_BK, ix_lds);
}

// Both expert GEMMs over a block map of 32 MI rows a tile, or IX_DECLINED. The weights are loaded past the caches (ix_dma16) while
// nearly every expert has one tile; SHARED: the height is also used where experts have two, with weight loads that cache.
template <int MI, bool SHARED>
static int ix_moe_experts_bands(const bf16_t* x, long ldx, int T, long rows, const int* sorted_token,
                                const float* permuted_prob, const bf16_t* W1, const bf16_t* W2, const int* meta,
                                long max_tiles, bf16_t* inter, bf16_t* out, int Hd, int F, hipStream_t st) {
  using C0 = IxBandCfg<MI, !SHARED>;
  using C1 = IxBandCfg<MI, true>;
  const long nb1 = F / 128, nb2 = Hd / 256;
  if (max_tiles * nb1 > 0x7fffffffL || max_tiles * nb2 > 0x7fffffffL) return IX_DECLINED;
  static bool attr_set = false;
  if (!attr_set) {
    for (const void* k : {(const void*)k_moe_fc1_glu_bands<C0>, (const void*)k_moe_fc1_glu_bands<C1>,
                          (const void*)k_moe_fc2_stream<C0>, (const void*)k_moe_fc2_stream<C1>})
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, C0::LDS_BYTES) != hipSuccess)
        return IX_ERR_LAUNCH;
    attr_set = true;
  }
  const bool once = rows <= 7 * C0::BM / 8 * (max_tiles - rows / C0::BM);
  hipLaunchKernelGGL(once ? k_moe_fc1_glu_bands<C1> : k_moe_fc1_glu_bands<C0>, dim3(IX_STREAM_WORKGROUPS), dim3(256),
                     C0::LDS_BYTES, st, x, ldx, T, (int)rows, sorted_token, permuted_prob, W1, meta, (int)max_tiles, inter, Hd,
                     F, (int)nb1);
  hipLaunchKernelGGL(once ? k_moe_fc2_stream<C1> : k_moe_fc2_stream<C0>, dim3(IX_STREAM_WORKGROUPS), dim3(256),
                     C0::LDS_BYTES, st, inter, W2, meta, (int)max_tiles, out, Hd, F, (int)nb2);
  return ix_launch_status();
}

// What the bands serve: Hd a multiple of 256 and F of 128 with enough k-tiles for the deferred epilogues, 32-bit byte offsets
// into the permutation's arrays, an expert's weight rows and a tile's output rows.
static inline bool ix_moe_bands_fit(long rows, long Hd, long F) {
  return Hd % 256 == 0 && Hd / IX_BK >= IxMoeFc1BandJob<IxBandCfg<3, false>>::NSK + 4 && F % 128 == 0 &&
         F / IX_BK >= IX_BAND_MIN_KT && rows < 0x20000000L && (F + 128) * Hd * 2 < 0x40000000L && Hd * 512 < 0x40000000L;
}

// ix_moe_bands_low.hip: 96 and 160 rows; ix_moe_bands_high.hip: 192
#define IX_MOE_BANDS_ARGS                                                                                              \
  int BM, const bf16_t *x, long ldx, int T, long rows, const int *sorted_token, const float *permuted_prob, const bf16_t *W1, \
      const bf16_t *W2, const int *meta, long max_tiles, bf16_t *inter, bf16_t *out, int Hd, int F, hipStream_t st
int ix_moe_experts_bands_low(IX_MOE_BANDS_ARGS);
int ix_moe_experts_bands_high(IX_MOE_BANDS_ARGS);
