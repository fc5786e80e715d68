// Pipeline G: pipeline F (ix_gemm_stream.h) for tiles of 32 MI rows x 256 columns, MI = 3 .. 7.
//
// The 256-row tile pays for 256 rows whatever it holds: 513 rows are three of them (a third of the matrix instructions
// work on padding), and an expert of 130 rows wastes half of one. Here the four waves of a workgroup stand side by side
// (one row of waves, 32 MI rows x 64 columns each), so a tile's height is any multiple of 32 that the accumulators hold.
// A phase has 2 MI matrix instructions; the fragment reads of the next one (MI + 2), the fetches and the pending tile's
// micro-steps are dealt over the slots behind them.
//
// The ring keeps three weight units of 32 KiB and, beside them, three activation units of 4 MI KiB (two from MI = 6 up:
// the LDS has no room for the third). A unit is free when its k-tile's last fragments are in registers, that is at the
// barrier in front of the k-tile's last phase; window w = that phase of k-tile w - 1 and the first three phases of k-tile
// w fetches W(w + 2) and X(w + LAX), LAX = units - 1, and the wait at its end leaves exactly those in flight that belong
// past k-tile w + 1. Same instruction, same K order, same roundings as every other pipeline.
//
// The job's interface is pipeline F's, except: micro-steps are numbered through the leading NSK k-tiles, 8 MI per k-tile;
// static constexpr bool is_store(i) says whether step i issues a vector-memory store; open_next() is called in the
// fourth-last k-tile and turn_offsets() in the window that first fetches the next tile's rows (one full window later at
// least: everything issued in open_next() has landed).
#pragma once
#include "ix_gemm_stream.h"

#define IX_BAND_MIN_KT (IX_STREAM_NSK + 4)

template <int MI_, bool W_ONCE_>
struct IxBandCfg {
  static constexpr bool W_ONCE = W_ONCE_;
  static constexpr int MI = MI_, NI = 2, WM = 1, WN = 4, NT = 256;
  static constexpr int BM = 32 * MI, BN = 256, TM = BM, TN = 64;
  static constexpr int X_CH = MI, W_CH = 8;  // 16-byte chunks a thread fetches per unit
  static constexpr int X_UNIT = BM * 128, W_UNIT = BN * 128, NW = 3;
  static constexpr int NX = NW * W_UNIT + 3 * X_UNIT <= 160 * 1024 ? 3 : 2;
  static constexpr int LDS_BYTES = NW * W_UNIT + NX * X_UNIT;
  static_assert(MI >= 3 && MI <= 7 && LDS_BYTES <= 160 * 1024, "the ring fits the LDS, the accumulators the registers");
};

// Slot (0 .. 8 MI - 1) of its window in which fetch f goes out. LAX = 2: 8 weight chunks, then MI activation chunks, spread
// evenly. LAX = 1: the activations are for the very next k-tile, so they take the first half, the weights the second.
template <int MI, int LAX>
__host__ __device__ constexpr int ix_band_fetch_slot(int f) {
  return LAX == 2 ? (2 * f + 1) * 8 * MI / (2 * (MI + 8)) : (f < MI ? 4 * f + 2 : 4 * MI + (2 * (f - MI) + 1) * MI / 4);
}
template <int MI, int LAX>
__host__ __device__ constexpr int ix_band_fetches_before(int slot) {
  int n = 0;
  while (n < MI + 8 && ix_band_fetch_slot<MI, LAX>(n) < slot) ++n;
  return n;
}
template <typename Job>
__host__ __device__ constexpr int ix_band_stores(int lo, int hi) {
  int n = 0;
  for (int i = lo; i < hi; ++i) n += Job::is_store(i) ? 1 : 0;
  return n;
}

template <typename Cfg, typename Job>
__device__ __forceinline__ void ix_gemm_bands(Job& job, int KT, char* lds) {
  constexpr int NT = Cfg::NT, MI = Cfg::MI, NSK = Job::NSK, NX = Cfg::NX, LAX = NX - 1, NF = MI + 8, PS = 2 * MI;
  constexpr int XB = Cfg::NW * Cfg::W_UNIT;  // the activation units follow the weight units
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t lds_base = __builtin_amdgcn_readfirstlane(ix_lds_addr(lds) + (wave * 64) * 16);

  if (!job.open_first()) return;
  ix_rsrc_t xr_c = job.nx_xr, wr_c = job.nx_wr, xr_n = xr_c, wr_n = wr_c;
  job.first_voffs();
  job.advance();

  const int frow = lane & 31, fg = lane >> 5;
  int x_foff[MI], w_foff[2];
#pragma unroll
  for (int i = 0; i < MI; ++i) x_foff[i] = ix_lds_off(i * 32 + frow, fg * 4);
#pragma unroll
  for (int i = 0; i < 2; ++i) w_foff[i] = ix_lds_off(wave * Cfg::TN + Job::w_frag_row(i, frow), fg * 4);
  // As in pipeline F: the weight fragments of a step are double-buffered, activation fragment i is overwritten right
  // after its last use.
  ix_bf16x8 fx[MI], fa[2], fb[2];
  ix_f32x16 acc[MI][2];
  const ix_f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  auto fetch_x = [&](auto jc, const ix_rsrc_t& rsrc, int t, int slot) {
    constexpr int j = decltype(jc)::value;
    ix_dma16<Job::DMA_IDLE>(rsrc, lds_base + XB + slot * Cfg::X_UNIT + j * NT * 16, job.template x_voff<j>(), t * (IX_BK * 2));
  };
  auto fetch_w = [&](auto jc, const ix_rsrc_t& rsrc, int t, int slot) {
    constexpr int j = decltype(jc)::value;
    ix_dma16<Job::DMA_IDLE, Cfg::W_ONCE>(rsrc, lds_base + slot * Cfg::W_UNIT + j * NT * 16, job.template w_voff<j>(),
                                         t * (IX_BK * 2));
  };
  // the fetches of window slot G: W(tw) of the tile behind wr into weight slot sw, X(tx) behind xr into slot sx
  auto fetches = [&](auto gc, const ix_rsrc_t& xr, const ix_rsrc_t& wr, int tx, int tw, int sx, int sw) {
    constexpr int LO = ix_band_fetches_before<MI, LAX>(decltype(gc)::value);
    constexpr int HI = ix_band_fetches_before<MI, LAX>(decltype(gc)::value + 1);
    ix_static_for<LO, HI>([&](auto fc) {
      constexpr int f = decltype(fc)::value;
      constexpr bool is_x = LAX == 2 ? f >= 8 : f < MI;
      if constexpr (is_x) fetch_x(std::integral_constant<int, LAX == 2 ? f - 8 : f>{}, xr, tx, sx);
      else fetch_w(std::integral_constant<int, LAX == 2 ? f : f - MI>{}, wr, tw, sw);
    });
  };

#define IXB_READ_X(XS, S, I) fx[I] = *reinterpret_cast<const ix_bf16x8*>((XS) + (x_foff[I] ^ ((S) << 4)))
#define IXB_READ_W(F, WS, S, I) F[I] = *reinterpret_cast<const ix_bf16x8*>((WS) + (w_foff[I] ^ ((S) << 4)))
  // One phase: 2 MI matrix instructions (mi = j / 2, ni = j % 2) on weight buffer FM; behind instructions 0 and 2 the weight
  // fragments of step S at (XS, WS) into FR, behind 2 i + 1 activation fragment i; window slots G0 + j and micro-steps
  // SLICE * 8 MI + PH * 2 MI + j.
#define IXB_PHASE(FM, FR, XS, WS, S, XR, WR, TX, TW, SX, SW, G0, PH, Z, SLICE)                                       \
  ix_static_for<0, PS>([&](auto jc) {                                                                                \
    constexpr int j = decltype(jc)::value;                                                                           \
    if constexpr (Z) acc[j >> 1][j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(FM[j & 1], fx[j >> 1], zero16, 0, 0, 0); \
    else acc[j >> 1][j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(FM[j & 1], fx[j >> 1], acc[j >> 1][j & 1], 0, 0, 0); \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
    if constexpr ((j & 1) == 1) IXB_READ_X(XS, S, j >> 1);                                                           \
    else if constexpr (j < 4) IXB_READ_W(FR, WS, S, j >> 1);                                                         \
    fetches(std::integral_constant<int, (G0) + j>{}, XR, WR, TX, TW, SX, SW);                                        \
    if constexpr ((SLICE) >= 0) job.template micro<((SLICE) < 0 ? 0 : (SLICE)) * 8 * MI + (PH) * PS + j>();          \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
  })

  auto wslot = [](int s) { return s >= Cfg::NW ? s - Cfg::NW : s; };
  auto xslot = [](int s) { return s >= NX ? s - NX : s; };
  // ---- the first tile: units of k-tiles 0 and (weights, and activations if LAX = 2) 1, then window 0's first phase
  ix_static_for<0, 8>([&](auto jc) { fetch_w(jc, wr_c, 0, 0); });
  ix_static_for<0, MI>([&](auto jc) { fetch_x(jc, xr_c, 0, 0); });
  ix_static_for<0, 8>([&](auto jc) { fetch_w(jc, wr_c, 1, 1); });
  if constexpr (LAX == 2) ix_static_for<0, MI>([&](auto jc) { fetch_x(jc, xr_c, 1, 1); });
  ix_static_for<0, PS>([&](auto gc) { fetches(gc, xr_c, wr_c, LAX, 2, LAX, 2); });
  constexpr int AHEAD = 8 + (LAX == 2 ? MI : 0);
  int cw = 0, cx = 0;  // slots of the k-tile's units
  __builtin_amdgcn_s_waitcnt(IX_VMCNT(AHEAD));  // k-tile 0 has landed (what window 0 has issued is on top)
  __syncthreads();
  ix_static_for<0, MI>([&](auto ic) { IXB_READ_X(lds + XB, 0, decltype(ic)::value); });
  ix_static_for<0, 2>([&](auto ic) { IXB_READ_W(fa, lds, 0, decltype(ic)::value); });

  auto ktile = [&](auto plan, int kt) {
    using P = decltype(plan);
    constexpr int TAIL = P::TAIL, SLICE = P::SLICE;
    constexpr bool ZERO = P::ZERO;
    if constexpr (TAIL == 4) {
      job.open_next();
      xr_n = job.nx_xr;
      wr_n = job.nx_wr;
    }
    // window kt: W(kt + 2), X(kt + LAX); window kt + 1 (the last phase): one further. Past the tile's end: the next tile's.
    constexpr bool WN0 = TAIL == 1 || TAIL == 2, WN1 = WN0 || TAIL == 3;
    constexpr bool XN0 = LAX == 2 ? WN0 : TAIL == 1, XN1 = LAX == 2 ? WN1 : WN0;
    const int tw0 = WN0 ? 2 - TAIL : kt + 2, tw1 = WN1 ? 3 - TAIL : kt + 3;
    const int tx0 = XN0 ? LAX - TAIL : kt + LAX, tx1 = XN1 ? LAX + 1 - TAIL : kt + LAX + 1;
    const char* ws = lds + cw * Cfg::W_UNIT;
    const char* xs = lds + XB + cx * Cfg::X_UNIT;
    const int fw = wslot(cw + 2), fxs = xslot(cx + LAX);
    IXB_PHASE(fa, fb, xs, ws, 1, (XN0 ? xr_n : xr_c), (WN0 ? wr_n : wr_c), tx0, tw0, fxs, fw, PS, 0, ZERO, SLICE);
    IXB_PHASE(fb, fa, xs, ws, 2, (XN0 ? xr_n : xr_c), (WN0 ? wr_n : wr_c), tx0, tw0, fxs, fw, 2 * PS, 1, false, SLICE);
    IXB_PHASE(fa, fb, xs, ws, 3, (XN0 ? xr_n : xr_c), (WN0 ? wr_n : wr_c), tx0, tw0, fxs, fw, 3 * PS, 2, false, SLICE);
    // Every fragment of this k-tile is in registers; k-tile kt + 1 has landed once only this window's fetches past it (and
    // the stores issued among them) are in flight: all NF of them, or the eight weight chunks and the stores of the two
    // phases that issue them.
    constexpr int S0 = (SLICE < 0 ? 0 : SLICE) * 8 * MI;
    constexpr int NST = SLICE < 0 ? 0 : (LAX == 2 ? ix_band_stores<Job>(S0, S0 + 3 * PS) : ix_band_stores<Job>(S0 + PS, S0 + 3 * PS));
    __builtin_amdgcn_s_waitcnt(IX_VMCNT((LAX == 2 ? NF : 8) + NST) & 0xF0FF);  // also lgkmcnt(0)
    __syncthreads();
    if constexpr (TAIL == 1 + LAX) job.turn_offsets();  // the current tile has made its last fetch through them
    const int gw = cw, gx = cx;  // the units this k-tile leaves
    cw = wslot(cw + 1);
    cx = xslot(cx + 1);
    const char* ws1 = lds + cw * Cfg::W_UNIT;
    const char* xs1 = lds + XB + cx * Cfg::X_UNIT;
    IXB_PHASE(fb, fa, xs1, ws1, 0, (XN1 ? xr_n : xr_c), (WN1 ? wr_n : wr_c), tx1, tw1, gx, gw, 0, 3, false, SLICE);
  };

  for (;;) {
    ix_static_for<0, NSK>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      ktile(IxKtPlan<s, s == 0, 0>{}, s);
    });
    for (int kt = NSK; kt < KT - 4; ++kt) ktile(IxKtPlan<-1, false, 0>{}, kt);
    ktile(IxKtPlan<-1, false, 4>{}, KT - 4);
    ktile(IxKtPlan<-1, false, 3>{}, KT - 3);
    ktile(IxKtPlan<-1, false, 2>{}, KT - 2);
    ktile(IxKtPlan<-1, false, 1>{}, KT - 1);
    asm volatile("s_nop 15\n\ts_nop 15");  // the matrix pipeline has drained before the accumulators are read by hand
    job.drain(acc);
    if (!job.has_next) break;
    job.advance();
    xr_c = xr_n;
    wr_c = wr_n;
  }
#undef IXB_PHASE
#undef IXB_READ_X
#undef IXB_READ_W
  __builtin_amdgcn_s_waitcnt(IX_VMCNT(0));
  ix_static_for<0, NSK * 8 * MI>([&](auto qc) { job.template micro<decltype(qc)::value>(); });
}
