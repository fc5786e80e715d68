// GatedDeltaNet: the gated delta-rule scan, its l2norm/gating preparation and the causal
// depthwise short conv.
//
// Scan (one function for varlen prefill and T=1 decode; reference call sites
// skyrl/backends/skyrl_train/isoexec/ops/gdn/gdn_ops.py:400-441 and :513-558):
//   per (sequence, value head hv), state S [V, K] fp32, for each token t in order
//     S      <- S * exp(g_t)
//     kv[v]   = sum_k S[v,k] * k_t[k]
//     d[v]    = (v_t[v] - kv[v]) * beta_t
//     S[v,k] <- S[v,k] + d[v] * k_t[k]
//     o_t[v]  = sum_k S[v,k] * (q_t[k] * scale)
//   state loaded from pool row idx[n,0], stored to pool row idx[n,t] after token t when that
//   index is > 0; a sequence whose idx[n,0] <= 0 is skipped (its outputs are written as 0).
//
// Each state row S[v,:] evolves independently, so the work is N*HV*V row recurrences. A row is
// owned by KS = K/8 consecutive lanes, lane s holding k = 8s..8s+7 in registers for the whole
// sequence. The two dot products use one fixed order: in-lane, two fused-multiply-add chains
// (even k, odd k) joined by one add; across the KS lanes, the adjacent-pairwise tree. The
// same device function runs for every token of a prefill and for a decode step, and a "chunk"
// is only how many tokens of q/k/v/g/beta are staged per LDS fill, so chunk length, the
// prefill/decode split and batch composition cannot move a bit.
#include "ix_common.h"
#include "../../include/isoexec_hip.h"

__device__ __forceinline__ float ix_ld(const float* p) { return *p; }
__device__ __forceinline__ float ix_ld(const bf16_t* p) { return ix_bf2f(*p); }
__device__ __forceinline__ void ix_st(float* p, float v) { *p = v; }
__device__ __forceinline__ void ix_st(bf16_t* p, float v) { *p = ix_f2bf(v); }

// dot of the lane's 8-element slices: (chain over k = 0,2,4,6) + (chain over k = 1,3,5,7)
__device__ __forceinline__ float ix_dot8(const float (&s)[8], const float (&x)[8]) {
  float pa = s[0] * x[0];
  float pb = s[1] * x[1];
  pa = __builtin_fmaf(s[2], x[2], pa);
  pb = __builtin_fmaf(s[3], x[3], pb);
  pa = __builtin_fmaf(s[4], x[4], pa);
  pb = __builtin_fmaf(s[5], x[5], pb);
  pa = __builtin_fmaf(s[6], x[6], pa);
  pb = __builtin_fmaf(s[7], x[7], pb);
  return pa + pb;
}

// One token of one state-row slice. Returns o (valid in every lane of the row's group).
template <int KS>
__device__ __forceinline__ float ix_gdn_step(float (&S)[8], const float (&kk)[8], const float (&qs)[8], float vv,
                                             float eg, float bt) {
#pragma unroll
  for (int i = 0; i < 8; ++i) S[i] = S[i] * eg;
  const float kv = ix_lane_tree<KS>(ix_dot8(S, kk));
  const float d = (vv - kv) * bt;
#pragma unroll
  for (int i = 0; i < 8; ++i) S[i] = __builtin_fmaf(d, kk[i], S[i]);
  return ix_lane_tree<KS>(ix_dot8(S, qs));
}

// RPL state rows per lane group: lane group r of the workgroup owns rows r, r + 256/KS, ... Each row is
// computed exactly as with RPL = 1 (same lanes per row, same order); holding several rows per lane only
// shares the k/q fetch and gives the scheduler independent chains to interleave.
template <int KS, int RPL, typename TIO>
__global__ __launch_bounds__(256) void k_gdn_scan(const TIO* __restrict__ q, const TIO* __restrict__ k,
                                                  const TIO* __restrict__ v, const float* __restrict__ g,
                                                  const TIO* __restrict__ beta, TIO* __restrict__ o,
                                                  float* __restrict__ state, const int* __restrict__ cu,
                                                  const int* __restrict__ sidx, long sidx_stride, long q_pitch,
                                                  long k_pitch, long v_pitch, int H, int HV, int V, float scale,
                                                  int TT, unsigned xcd_total) {
  constexpr int K = KS * 8;
  constexpr int RW = 256 / KS;   // state rows per pass over the lanes
  constexpr int R = RW * RPL;    // state rows per workgroup
  extern __shared__ __align__(16) char ix_lds[];
  float* kf = reinterpret_cast<float*>(ix_lds);  // [TT][K]
  float* qf = kf + TT * K;                       // [TT][K], pre-scaled
  float* vf = qf + TT * K;                       // [TT][R]
  float* of = vf + TT * R;                       // [TT][R]
  float* egf = of + TT * R;                      // [TT]
  float* btf = egf + TT;                         // [TT]
  int* sif = reinterpret_cast<int*>(btf + TT);   // [TT]

  const int VB = V / R;
  long bid = blockIdx.x;
  {
    unsigned pos;
    if (!ix_xcd_run_position(blockIdx.x, xcd_total, &pos)) return;
    bid = pos;
  }
  const int vb = (int)(bid % VB);
  bid /= VB;
  const int hv = (int)(bid % HV);
  const int n = (int)(bid / HV);
  const int h = hv / (HV / H);
  const int tid = threadIdx.x;
  const int sub = tid % KS, r = tid / KS;
  const int vrow = vb * R + r;  // row of pass 0; pass j adds j * RW

  const int t_begin = cu[n], t_end = cu[n + 1];
  const int len = t_end - t_begin;
  if (len <= 0) return;
  // Stride 0: one row per sequence, loaded at the first token and stored once after the last.
  const long sbase = sidx_stride == 0 ? (long)n : (long)n * sidx_stride;
  const int row0 = sidx[sbase];
  if (row0 <= 0) {  // null lane: no state, outputs defined as zero
    if (!o) return;
    for (int i = tid; i < len * R; i += 256) {
      const int tt = i / R, rr = i % R;
      ix_st(o + ((long)(t_begin + tt) * HV + hv) * V + vb * R + rr, 0.0f);
    }
    return;
  }

  // q and k rows can be fetched 8 elements at a time when every row start is 16/32-byte aligned
  constexpr long AL = 16 * sizeof(TIO) / 2;
  const bool vec_qk = (q_pitch % 8 == 0) && (k_pitch % 8 == 0) && ((uintptr_t)q % AL == 0) && ((uintptr_t)k % AL == 0);
  float S[RPL][8];
#pragma unroll
  for (int j = 0; j < RPL; ++j) {
    const float* sp = state + (((long)row0 * HV + hv) * V + vrow + j * RW) * K + sub * 8;
    const float4 a = *reinterpret_cast<const float4*>(sp);
    const float4 b = *reinterpret_cast<const float4*>(sp + 4);
    S[j][0] = a.x; S[j][1] = a.y; S[j][2] = a.z; S[j][3] = a.w;
    S[j][4] = b.x; S[j][5] = b.y; S[j][6] = b.z; S[j][7] = b.w;
  }

  for (int t0 = 0; t0 < len; t0 += TT) {
    const int nt = min(TT, len - t0);
    __syncthreads();
    if (vec_qk) {  // 8 elements (16 bytes) per load
      for (int i = tid; i < nt * (K / 8); i += 256) {
        const int tt = i / (K / 8), kk = (i % (K / 8)) * 8;
        const long tok = t_begin + t0 + tt;
        float a[8], b[8];
        ix_load8(k + tok * k_pitch + h * K + kk, 8, true, 0.0f, a);
        ix_load8(q + tok * q_pitch + h * K + kk, 8, true, 0.0f, b);
        float* kd = kf + tt * K + kk;
        float* qd = qf + tt * K + kk;
        *reinterpret_cast<float4*>(kd) = make_float4(a[0], a[1], a[2], a[3]);
        *reinterpret_cast<float4*>(kd + 4) = make_float4(a[4], a[5], a[6], a[7]);
        *reinterpret_cast<float4*>(qd) = make_float4(b[0] * scale, b[1] * scale, b[2] * scale, b[3] * scale);
        *reinterpret_cast<float4*>(qd + 4) = make_float4(b[4] * scale, b[5] * scale, b[6] * scale, b[7] * scale);
      }
    } else {
      for (int i = tid; i < nt * K; i += 256) {
        const int tt = i / K, kk = i % K;
        const long tok = t_begin + t0 + tt;
        kf[i] = ix_ld(k + tok * k_pitch + h * K + kk);
        qf[i] = ix_ld(q + tok * q_pitch + h * K + kk) * scale;
      }
    }
    for (int i = tid; i < nt * R; i += 256) {
      const int tt = i / R, rr = i % R;
      vf[i] = ix_ld(v + (long)(t_begin + t0 + tt) * v_pitch + (long)hv * V + vb * R + rr);
    }
    for (int i = tid; i < nt; i += 256) {
      const long src = (long)(t_begin + t0 + i) * HV + hv;
      egf[i] = ix_exp(g[src]);
      btf[i] = ix_ld(beta + src);
      sif[i] = sidx_stride == 0 ? (t0 + i == len - 1 ? row0 : 0) : sidx[sbase + t0 + i];
    }
    __syncthreads();
    auto token = [&](int tt) {
      float kk[8], qs[8];
      {
        const float4 a = *reinterpret_cast<const float4*>(kf + tt * K + sub * 8);
        const float4 b = *reinterpret_cast<const float4*>(kf + tt * K + sub * 8 + 4);
        kk[0] = a.x; kk[1] = a.y; kk[2] = a.z; kk[3] = a.w; kk[4] = b.x; kk[5] = b.y; kk[6] = b.z; kk[7] = b.w;
        const float4 c = *reinterpret_cast<const float4*>(qf + tt * K + sub * 8);
        const float4 d = *reinterpret_cast<const float4*>(qf + tt * K + sub * 8 + 4);
        qs[0] = c.x; qs[1] = c.y; qs[2] = c.z; qs[3] = c.w; qs[4] = d.x; qs[5] = d.y; qs[6] = d.z; qs[7] = d.w;
      }
      const float eg = egf[tt], bt = btf[tt];
      float ov[RPL];
#pragma unroll
      for (int j = 0; j < RPL; ++j) ov[j] = ix_gdn_step<KS>(S[j], kk, qs, vf[tt * R + j * RW + r], eg, bt);
      if (sub == 0) {
#pragma unroll
        for (int j = 0; j < RPL; ++j) of[tt * R + j * RW + r] = ov[j];
      }
    };
    auto store_state = [&](int si) {
#pragma unroll
      for (int j = 0; j < RPL; ++j) {
        float* sp = state + (((long)si * HV + hv) * V + vrow + j * RW) * K + sub * 8;
        *reinterpret_cast<float4*>(sp) = make_float4(S[j][0], S[j][1], S[j][2], S[j][3]);
        *reinterpret_cast<float4*>(sp + 4) = make_float4(S[j][4], S[j][5], S[j][6], S[j][7]);
      }
    };
    if (sidx_stride == 0) {
      // one store, after the sequence's last token: the token loop carries no per-token check
#pragma unroll 4
      for (int tt = 0; tt < nt; ++tt) token(tt);
      if (t0 + nt == len) store_state(row0);
    } else {
      for (int tt = 0; tt < nt; ++tt) {
        token(tt);
        const int si = sif[tt];
        if (si > 0) store_state(si);
      }
    }
    __syncthreads();
    if (o) {
      for (int i = tid; i < nt * R; i += 256) {
        const int tt = i / R, rr = i % R;
        ix_st(o + ((long)(t_begin + t0 + tt) * HV + hv) * V + vb * R + rr, of[i]);
      }
    }
  }
}

// ---- the same scan with a state row held by FOUR lanes and updated by the matrix pipe (K = 128) ----------------
// Lanes r, r + 16, r + 32, r + 48 of a wave own state rows r and r + 16 of the wave's 32, lane group g = lane / 16 the
// elements k = 32 g .. 32 g + 31 of both: 64 state floats per lane. The row's arithmetic is that of k_gdn_scan statement
// for statement -- per 8-element slice the same two multiply-add chains and their join (ix_dot8), the adjacent-pairwise
// tree over the 16 slice sums, here two levels inside the lane, one across neighbouring lane groups and one across the
// wave's halves -- so the two kernels agree bit for bit (a NaN's payload aside), and which one runs is a staging choice like the time
// tile.
// The rank-one update S += d k is four v_mfma_f32_16x16x1_4b_f32: state rows are the columns (B = d), the elements of k the
// rows (A, one value per lane), S the accumulator, whose register layout is the one above. With one product per element
// that instruction is a fused multiply-add, rounded once, subnormals kept (a million operands over the whole range against fmaf in
// ix_selfcheck.hip: every bit but a NaN's payload); of the four multiply-adds per element and token one leaves the vector pipe, which bounds
// this kernel: 240 vector and matrix instructions per token for a wave's 32 rows. Two rows per lane, and not one with 64
// elements, because every lane reads all its elements of k and q from LDS for each token: 18 reads of a wave instead of 34.
// 64 x 2560 tokens, 32 heads: 10.1 ms on the vector pipe alone (a row held by two lanes), 8.9 ms this way.
// Compact state form only (one pool row per sequence, stored after the last token; without a pool the sequences start
// from zero and nothing is stored).
#define IX_GDN_SORT_MAX 256  // sequences a workgroup ranks by length
// The sequence of rank `n` when sequences are taken longest first (ties in packed order), so that the long ones do not
// start last: every workgroup of a launch over 2..IX_GDN_SORT_MAX sequences ranks them itself, one per thread. `lens`:
// IX_GDN_SORT_MAX + 1 ints of LDS, free again on return.
__device__ __forceinline__ int ix_gdn_nth_longest(const int* __restrict__ cu, int N, int n, int* lens) {
  if (N < 2 || N > IX_GDN_SORT_MAX) return n;
  const int tid = threadIdx.x;
  const int mine = tid < N ? cu[tid + 1] - cu[tid] : 0;
  if (tid < N) lens[tid] = mine;
  __syncthreads();
  int rank = 0;
  for (int j = 0; j < N; ++j) rank += (lens[j] > mine || (lens[j] == mine && j < tid)) ? 1 : 0;
  if (tid < N && rank == n) lens[IX_GDN_SORT_MAX] = tid;
  __syncthreads();
  const int r = lens[IX_GDN_SORT_MAX];
  __syncthreads();
  return r;
}
__device__ __forceinline__ float ix_add_halves(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);  // (own half) + (other half) or the reverse: same bits
}
// Two sums over the wave's four groups of sixteen lanes, (0 + 1) + (2 + 3): groups 0 and 2 return a's, 1 and 3 b's.
__device__ __forceinline__ float ix_add_groups2(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return ix_add_halves(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}
typedef float ix_f32x16 __attribute__((ext_vector_type(16)));
// A lane group's 32 elements of a token's k or q in LDS. The groups' elements stand 36 floats apart, so that their reads fall
// on different banks; a token takes IX_QUAD_KP floats.
#define IX_QUAD_KP 140
__device__ __forceinline__ int ix_quad_at(int k) { return k + (k >> 5) * 4; }
__device__ __forceinline__ void ix_quad_load(const float* row, int grp, float (&x)[32]) {
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float4 a = *reinterpret_cast<const float4*>(row + 36 * grp + 4 * c);
    x[4 * c] = a.x; x[4 * c + 1] = a.y; x[4 * c + 2] = a.z; x[4 * c + 3] = a.w;
  }
}
// The lane's four slice sums of one state row, and the two levels of the row's tree that run inside the lane.
__device__ __forceinline__ float ix_quad_dot(const ix_f32x16 (&S)[2], const float (&x)[32]) {
  float part[4];
#pragma unroll
  for (int sl = 0; sl < 4; ++sl) {
    float ss[8], xs[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ss[i] = S[sl >> 1][8 * (sl & 1) + i];
      xs[i] = x[8 * sl + i];
    }
    part[sl] = ix_dot8(ss, xs);
  }
  return (part[0] + part[1]) + (part[2] + part[3]);
}

template <typename TIO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void k_gdn_scan_quads(const TIO* __restrict__ q, const TIO* __restrict__ k, const TIO* __restrict__ v,
                      const float* __restrict__ g, const TIO* __restrict__ beta, TIO* __restrict__ o,
                      float* __restrict__ state, const int* __restrict__ cu, const int* __restrict__ sidx,
                      long q_pitch, long k_pitch, long v_pitch, int N, int H, int HV, int V, float scale, int TT,
                      const bf16_t* __restrict__ gate, long gate_stride_t, const bf16_t* __restrict__ norm_w,
                      float norm_eps, int zero_centered) {
  constexpr int K = 128;
  constexpr int R = 128;  // state rows per workgroup: 4 waves x 32 rows
  constexpr int Q = IX_QUAD_KP, VAT = 2 * IX_QUAD_KP, OAT = VAT + R, EAT = OAT + R, REC = EAT + 4;
  extern __shared__ __align__(16) char ix_lds[];
  float* rec = reinterpret_cast<float*>(ix_lds);  // a token: k, q pre-scaled [IX_QUAD_KP each], v [R], o [R], exp(g), beta

  const int VB = V / R;
  long bid = blockIdx.x;
  const int vb = (int)(bid % VB);
  bid /= VB;
  const int hv = (int)(bid % HV);
  const int n = ix_gdn_nth_longest(cu, N, (int)(bid / HV), reinterpret_cast<int*>(ix_lds));
  const int h = hv / (HV / H);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int grp = lane >> 4;
  const int r = wave * 32 + (lane & 31);  // the row whose v, d and output this lane has

  const int t_begin = cu[n], t_end = cu[n + 1];
  const int len = t_end - t_begin;
  if (len <= 0) return;
  const int row0 = sidx ? sidx[n] : 1;
  // What leaves for the nt tokens of the tile at t0 whose outputs stand in `of`: the outputs themselves, or, with a gate,
  // the layer's gated output norm of them (ix_gated_out_norm: RMSNorm over the head's V = 128 values, bf16(1 + w),
  // silu(gate)) instead of a launch that reads them back. A token's head is sixteen consecutive threads of eight
  // values, k_rmsnorm_reg<16, 1, 1>'s layout, and the statements are its statements on the bf16 values this kernel
  // would have stored. V == 128 there (one row block per head).
  auto emit = [&](int t0, int nt) __attribute__((always_inline)) {
    if (gate) {
      for (int i0 = 0; i0 < nt * 16; i0 += 256) {
        const int i = i0 + tid;
        const bool live_row = i < nt * 16;
        const int tt = live_row ? i >> 4 : nt - 1, sub = i & 15;  // rows past the tile run the shuffles, never store
        const long tok = t_begin + t0 + tt;
        // The roundings inside the chain are the hardware pack-convert's (ix_rbf2_hw): it differs from ix_rbf on NaNs
        // only, a NaN stays a NaN through every operation below whatever its payload, and the values that are stored
        // get their NaNs made canonical (ix_pack_bf2_canon_hw) -- the stored bits are the ix_rbf chain's. This kernel
        // is bound by vector issue, so the twenty-odd instructions less per value are time.
        float xv[8], wv[8], gv[8], acc[8];
        uint32_t op[4];
        ix_unpack8(*reinterpret_cast<const uint4*>(gate + tok * gate_stride_t + (long)hv * V + sub * 8), gv);
        ix_unpack8(*reinterpret_cast<const uint4*>(norm_w + sub * 8), wv);
#pragma unroll
        for (int j = 0; j < 8; j += 2)  // the scan's output is a bf16 tensor
          ix_rbf2_hw(rec[tt * REC + OAT + sub * 8 + j], rec[tt * REC + OAT + sub * 8 + j + 1], xv[j], xv[j + 1]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float sq = xv[j] * xv[j];
          acc[j] = 0.0f + sq;
        }
        const float ssum = ix_lane_tree<16>(ix_tree8(acc));
        const float ms = ssum / 128.0f;
        const float rstd = ix_rsqrt_ieee(ms + norm_eps);
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          float nb0, nb1, g0 = wv[j], g1 = wv[j + 1], y0, y1;
          ix_rbf2_hw(xv[j] * rstd, xv[j + 1] * rstd, nb0, nb1);
          if (zero_centered) ix_rbf2_hw(1.0f + wv[j], 1.0f + wv[j + 1], g0, g1);
          ix_rbf2_hw(nb0 * g0, nb1 * g1, y0, y1);
          op[j >> 1] = ix_pack_bf2_canon_hw(y0 * ix_silu_div(gv[j]), y1 * ix_silu_div(gv[j + 1]));
        }
        if (live_row)
          *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(o) + (tok * HV + hv) * V + sub * 8) =
              make_uint4(op[0], op[1], op[2], op[3]);
      }
    } else {
      for (int i = tid; i < nt * R; i += 256) {
        const int tt = i / R, rr = i % R;
        ix_st(o + ((long)(t_begin + t0 + tt) * HV + hv) * V + vb * R + rr, rec[tt * REC + OAT + rr]);
      }
    }
  };
  if (row0 <= 0) {  // null lane: no state, outputs defined as zero (and what the norm makes of zeros)
    if (!o) return;
    for (int i = tid; i < TT * R; i += 256) rec[i / R * REC + OAT + i % R] = 0.0f;
    __syncthreads();
    for (int t0 = 0; t0 < len; t0 += TT) emit(t0, min(TT, len - t0));
    return;
  }
  constexpr long AL = 16 * sizeof(TIO) / 2;
  const bool vec_qk = (q_pitch % 8 == 0) && (k_pitch % 8 == 0) && ((uintptr_t)q % AL == 0) && ((uintptr_t)k % AL == 0);
  // S[j][c][i]: row wave * 32 + 16 j + lane % 16, k = 32 grp + 16 c + i
  ix_f32x16 S[2][2];
  float* srow = state + (((long)row0 * HV + hv) * V + vb * R + wave * 32 + (lane & 15)) * K + 32 * grp;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float4 a =
          state ? *reinterpret_cast<const float4*>(srow + 16 * j * K + 4 * c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      ix_f32x16& d = S[j][c >> 2];
      const int i = 4 * (c & 3);
      d[i] = a.x; d[i + 1] = a.y; d[i + 2] = a.z; d[i + 3] = a.w;
    }
  }
  // the element of k that this lane hands to the update's first instruction (the second one's: 16 further)
  const int ka = 36 * ((lane & 15) >> 2) + 4 * grp + (lane & 3);
  // both rows' dot products with 32 elements of k or q: groups 0 and 2 have the first row's, 1 and 3 the second's
  auto dots = [&](const float (&x)[32]) __attribute__((always_inline)) {
    return ix_add_groups2(ix_quad_dot(S[0], x), ix_quad_dot(S[1], x));
  };

  for (int t0 = 0; t0 < len; t0 += TT) {
    const int nt = min(TT, len - t0);
    __syncthreads();
    if (vec_qk) {  // 8 elements (16 bytes) per load
      for (int i = tid; i < nt * (K / 8); i += 256) {
        const int tt = i / (K / 8), kk = (i % (K / 8)) * 8;
        const long tok = t_begin + t0 + tt;
        float a[8], b[8];
        ix_load8(k + tok * k_pitch + h * K + kk, 8, true, 0.0f, a);
        ix_load8(q + tok * q_pitch + h * K + kk, 8, true, 0.0f, b);
        float* kd = rec + tt * REC + ix_quad_at(kk);
        float* qd = kd + Q;
        *reinterpret_cast<float4*>(kd) = make_float4(a[0], a[1], a[2], a[3]);
        *reinterpret_cast<float4*>(kd + 4) = make_float4(a[4], a[5], a[6], a[7]);
        *reinterpret_cast<float4*>(qd) = make_float4(b[0] * scale, b[1] * scale, b[2] * scale, b[3] * scale);
        *reinterpret_cast<float4*>(qd + 4) = make_float4(b[4] * scale, b[5] * scale, b[6] * scale, b[7] * scale);
      }
    } else {
      for (int i = tid; i < nt * K; i += 256) {
        const int tt = i / K, kk = i % K;
        const long tok = t_begin + t0 + tt;
        float* at = rec + tt * REC + ix_quad_at(kk);
        at[0] = ix_ld(k + tok * k_pitch + h * K + kk);
        at[Q] = ix_ld(q + tok * q_pitch + h * K + kk) * scale;
      }
    }
    for (int i = tid; i < nt * R; i += 256) {
      const int tt = i / R, rr = i % R;
      rec[tt * REC + VAT + rr] = ix_ld(v + (long)(t_begin + t0 + tt) * v_pitch + (long)hv * V + vb * R + rr);
    }
    for (int i = tid; i < nt; i += 256) {
      const long src = (long)(t_begin + t0 + i) * HV + hv;
      rec[i * REC + EAT] = ix_exp(g[src]);
      rec[i * REC + EAT + 1] = ix_ld(beta + src);
    }
    __syncthreads();
    auto token = [&](int tt) __attribute__((always_inline)) {
      float* at = rec + tt * REC;
      const float eg = at[EAT], bt = at[EAT + 1], vv = at[VAT + r];
      float x[32];  // this lane group's elements of k, later of q
      ix_quad_load(at, grp, x);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 16; ++i) S[j][c][i] = S[j][c][i] * eg;
      const float d = (vv - dots(x)) * bt;
      // groups 0 and 2 have the first row's d, 1 and 3 the second's: each to all four
      const auto dd = __builtin_amdgcn_permlane16_swap(__float_as_uint(d), __float_as_uint(d), false, false);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float ke = at[ka + 16 * c];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          S[j][c] = __builtin_amdgcn_mfma_f32_16x16x1f32(ke, __uint_as_float(dd[j]), S[j][c], 0, 0, 0);
      }
      ix_quad_load(at + Q, grp, x);
      const float ov = dots(x);
      at[OAT + r] = ov;  // both halves of the wave have it
    };
    int tt = 0;
    for (; tt + 4 <= nt; tt += 4) {  // four tokens at fixed distances from one set of addresses
#pragma unroll
      for (int u = 0; u < 4; ++u) token(tt + u);
    }
    for (; tt < nt; ++tt) token(tt);
    if (state && t0 + nt == len) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const ix_f32x16& a = S[j][c >> 2];
          const int i = 4 * (c & 3);
          *reinterpret_cast<float4*>(srow + 16 * j * K + 4 * c) = make_float4(a[i], a[i + 1], a[i + 2], a[i + 3]);
        }
    }
    __syncthreads();
    if (o) emit(t0, nt);
  }
}

// ---- prefill of few sequences: the walk ---------------------------------------------------------------------
// One sequence has HV * V row recurrences and a token's step is a chain through each of them (decay, multiply-adds, tree,
// update): with few sequences the time is tokens x the latency of that chain, and with some more the vector issue of the
// waves that share a SIMD. So the layout is the sixteen-lane one (one sequence of HV = 32, V = 128 heads is then
// exactly one wave per SIMD), and everything that is not the chain is kept out of its way:
//   * tiles of 16 tokens, staged twice in LDS: the next tile's global loads are issued before this tile's tokens and
//     written to LDS after them; one barrier per tile;
//   * hardly an LDS store between a tile's tokens (an LDS load may not pass one): a token's output is the same in all lanes of
//     its row, so lane tt keeps token tt's and the row's lanes store together, once every L tokens;
//   * sixteen tokens of straight-line code, so the output's tree runs in the shadow of the next token's decay and dot;
//   * LONE, at a workgroup or two per CU: a fifth wave stages the tiles and writes the outputs out, so that the four others
//     meet nothing but their tokens and the barrier (a fifth of the walk at one wave per SIMD, which waits for its own every
//     instruction: 1147 -> 988 us for 8192 tokens, 121 ns a token);
//   * E = 4, where SIMDs would stand idle: a slice's two chains in two lanes, joined by the tree's first level. A token is then
//     29 vector instructions of a wave instead of 45 (256 tokens at K = 64: 33 -> 24 us).
// The statements per token are ix_gdn_step's: same bits as k_gdn_scan and k_gdn_scan_quads.
// Sequences are taken longest first when there are 2..256 of them (ranked by every workgroup from cu), and a sequence's
// workgroups are spread over all XCDs with the row blocks of a key head on one of them.
// CPR: the boundary form (gdn_cpr.py:296-319). Two states walk together: the fp32 chain, and the running state, which
// restarts from the chain rounded to the io type at every multiple of `chunk` tokens and makes the outputs. The pass that
// first computes every boundary state, its pool, and the second pass over all tokens are then not there at all.
// Measured (HV = 32, V = K = 128, bf16), k_gdn_scan / walk: without LONE one sequence of 8192 tokens 1990 / 1129 us (138 ns a
// token; vector issue alone would be 75), five of 33..1203 tokens 883 / 247, 8 x 1000 1330 / 667; boundary form of nine sequences
// of 120..1500 tokens, boundary pass + segmented scan / walk: 3900 / 975. With first and second halves of the 8-element
// slices apart in LDS a 16-byte read of sixteen lanes is one contiguous row (8 x 1000: 714 -> 667).
__device__ __forceinline__ float ix_wire(float x, const bf16_t*) { return ix_rbf(x); }
__device__ __forceinline__ float ix_wire(float x, const float*) { return x; }

// dot of a lane's slice in the canonical order: eight elements, two chains joined; four elements, one of the two chains (the
// join is then the first level of the lane tree).
template <int E>
__device__ __forceinline__ float ix_dot_slice(const float (&s)[E], const float (&x)[E]) {
  if constexpr (E == 8) {
    return ix_dot8(s, x);
  } else {
    float p = s[0] * x[0];
    p = __builtin_fmaf(s[1], x[1], p);
    p = __builtin_fmaf(s[2], x[2], p);
    return __builtin_fmaf(s[3], x[3], p);
  }
}

template <int K, int E, int RPL, typename TIO, bool CPR, bool LONE>
__global__ __launch_bounds__(LONE ? 320 : 256) void k_gdn_walk(const TIO* __restrict__ q, const TIO* __restrict__ k,
                                                  const TIO* __restrict__ v, const float* __restrict__ g,
                                                  const TIO* __restrict__ beta, TIO* __restrict__ o,
                                                  float* __restrict__ state, const int* __restrict__ cu,
                                                  const int* __restrict__ sidx, long q_pitch, long k_pitch,
                                                  long v_pitch, int N, int H, int HV, int V, float scale, int chunk) {
  constexpr int T = K == 256 ? 8 : 16;           // tokens per tile (K = 256: half as many, for the LDS)
  constexpr int L = K / E;                       // lanes per row
  constexpr int RW = 256 / L;
  constexpr int R = RW * RPL;
  constexpr int G8 = K / 8;
  constexpr int QK = 2 * T * G8;                 // 8-element groups of k and q in a tile
  constexpr int ST = LONE ? 64 : 256;            // threads that stage
  constexpr int QC = (QK + ST - 1) / ST;         // groups per staging thread
  constexpr int VC = (T * R + ST - 1) / ST;      // v elements per staging thread
  __shared__ __align__(16) float kq[2][2][T][K];  // [buffer][k, q * scale][token]
  __shared__ float vf[2][T][R];
  __shared__ float of[2][T][R];
  __shared__ float2 eb[2][T];                    // exp(g), beta

  const int VB = V / R;
  const int per_seq = HV * VB;
  const int tid = threadIdx.x;
  int n, w;
  {
    const unsigned bid = blockIdx.x;
    if ((per_seq & 7) == 0) {  // hardware deals consecutive ids to the XCDs round-robin
      const unsigned per8 = (unsigned)per_seq >> 3;
      n = (int)((bid >> 3) / per8);
      w = (int)((bid & 7u) * per8 + (bid >> 3) % per8);
    } else {
      n = (int)(bid / (unsigned)per_seq);
      w = (int)(bid % (unsigned)per_seq);
    }
  }
  static_assert(sizeof(kq) >= (IX_GDN_SORT_MAX + 1) * sizeof(int), "the ranking uses the staging buffer");
  n = ix_gdn_nth_longest(cu, N, n, reinterpret_cast<int*>(&kq[0][0][0][0]));
  const int vb = w % VB;
  const int hv = w / VB;
  const int h = hv / (HV / H);
  const int t_begin = cu[n];
  const int len = cu[n + 1] - t_begin;
  if (len <= 0) return;
  const int row0 = sidx ? sidx[n] : 1;
  TIO* ob = o + (long)hv * V + vb * R;
  if (row0 <= 0) {  // null lane: no state, outputs defined as zero
    for (int i = tid; i < len * R; i += (int)blockDim.x) ix_st(ob + (long)(t_begin + i / R) * HV * V + i % R, 0.0f);
    return;
  }
  const int tiles = (len + T - 1) / T;

  const int lane = LONE ? tid - 256 : tid;       // among the staging threads
  IxRaw8<TIO> rq[QC];
  // raw, as loaded: a conversion here would wait for the loads that the tile's tokens are meant to cover
  TIO rv[VC], rb = 0;
  float rg = 0.0f;
  auto fetch = [&](int t0) __attribute__((always_inline)) {  // tokens past the end read the last one's values, unused
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const int i = lane + ST * c;
      if (QK % ST == 0 || i < QK) {
        const int e = i % (T * G8), isq = i / (T * G8);
        const long tok = t_begin + min(t0 + e / G8, len - 1);
        rq[c].load((isq ? q + tok * q_pitch : k + tok * k_pitch) + h * K + (e % G8) * 8);
      }
    }
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      const int i = lane + ST * c;
      if ((T * R) % ST == 0 || i < T * R) {
        const long tok = t_begin + min(t0 + i / R, len - 1);
        rv[c] = v[tok * v_pitch + (long)hv * V + vb * R + i % R];
      }
    }
    if (lane < T) {
      const long tok = t_begin + min(t0 + lane, len - 1);
      rg = g[tok * HV + hv];
      rb = beta[tok * HV + hv];
    }
  };
  auto commit = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const int i = lane + ST * c;
      if (QK % ST == 0 || i < QK) {
        const int e = i % (T * G8), isq = i / (T * G8);
        float x[8];
        rq[c].widen(x);
        const float m = isq ? scale : 1.0f;  // k * 1 is k
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = x[j] * m;
        if constexpr (E == 8) {  // first halves of all slices, then second halves: sixteen lanes read one contiguous row
          float* d = &kq[b][isq][e / G8][(e % G8) * 4];
          *reinterpret_cast<float4*>(d) = make_float4(x[0], x[1], x[2], x[3]);
          *reinterpret_cast<float4*>(d + K / 2) = make_float4(x[4], x[5], x[6], x[7]);
        } else {  // a slice's even elements, then its odd ones: one chain each
          float* d = &kq[b][isq][e / G8][(e % G8) * 8];
          *reinterpret_cast<float4*>(d) = make_float4(x[0], x[2], x[4], x[6]);
          *reinterpret_cast<float4*>(d + 4) = make_float4(x[1], x[3], x[5], x[7]);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      const int i = lane + ST * c;
      if ((T * R) % ST == 0 || i < T * R) vf[b][i / R][i % R] = ix_ld(&rv[c]);
    }
    if (lane < T) eb[b][lane] = make_float2(ix_exp(rg), ix_ld(&rb));
  };
  auto emit = [&](int t0, int nt, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      const int i = lane + ST * c;
      if (i < nt * R) ix_st(ob + (long)(t_begin + t0 + i / R) * HV * V + i % R, of[b][i / R][i % R]);
    }
  };
  if constexpr (LONE) {
    // The staging wave: as many barriers as the others. The branch is the same for a whole wave (256 is a multiple of 64); with the
    // wave number in a scalar register the compiler keeps both sides' values at once, and two workgroups no longer fit a CU (K = 256,
    // 3 x 1000 tokens 208 -> 300 us).
    if (tid >= 256) {
      fetch(0);
      commit(0);
      if (tiles > 1) fetch(T);
      __syncthreads();
      for (int i = 0; i < tiles; ++i) {
        const int b = i & 1;
        if (i + 1 < tiles) commit(b ^ 1);
        if (i + 2 < tiles) fetch((i + 2) * T);
        if (i > 0) emit((i - 1) * T, T, b ^ 1);
        __syncthreads();
      }
      emit((tiles - 1) * T, len - (tiles - 1) * T, (tiles - 1) & 1);
      return;
    }
    __builtin_amdgcn_s_setprio(2);  // in front of the staging wave, which has a tile's time for its share
  }

  const int sub = tid % L, r = tid / L;
  float S[RPL][E], C[CPR ? RPL : 1][E];
  const int kbase = E == 8 ? sub * 8 : (sub >> 1) * 8 + (sub & 1);
  // whole slices come and go 16 bytes at a time: one element at a time, 200 sequences of 9 tokens (K = V = 64, 32 heads) take
  // 120 us instead of 104
#pragma unroll
  for (int j = 0; j < RPL; ++j) {
    const float* sp = state + (((long)row0 * HV + hv) * V + vb * R + r + j * RW) * K + kbase;
    if constexpr (E == 4) {
#pragma unroll
      for (int i = 0; i < E; ++i) S[j][i] = state ? sp[i * 2] : 0.0f;
    } else if (state) {
      const float4 a = *reinterpret_cast<const float4*>(sp);
      const float4 b = *reinterpret_cast<const float4*>(sp + 4);
      S[j][0] = a.x; S[j][1] = a.y; S[j][2] = a.z; S[j][3] = a.w;
      S[j][4] = b.x; S[j][5] = b.y; S[j][6] = b.z; S[j][7] = b.w;
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) S[j][i] = 0.0f;
    }
    if constexpr (CPR) {
#pragma unroll
      for (int i = 0; i < E; ++i) C[j][i] = S[j][i];
    }
  }
  auto load_x = [&](const float* row, float (&x)[E]) __attribute__((always_inline)) {
    const float4 a = *reinterpret_cast<const float4*>(row + sub * 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    if constexpr (E == 8) {
      const float4 c = *reinterpret_cast<const float4*>(row + K / 2 + sub * 4);
      x[4] = c.x; x[5] = c.y; x[6] = c.z; x[7] = c.w;
    }
  };

  if constexpr (!LONE) {
    fetch(0);
    commit(0);
  }
  __syncthreads();
  for (int it = 0; it < tiles; ++it) {
    const int b = it & 1, t0 = it * T;
    const int nt = min(T, len - t0);
    if constexpr (!LONE) {
      if (it + 1 < tiles) fetch(t0 + T);
      if (it > 0) emit(t0 - T, T, b ^ 1);
    }
    if constexpr (CPR) {
      if (t0 % chunk == 0) {
#pragma unroll
        for (int j = 0; j < RPL; ++j)
#pragma unroll
          for (int i = 0; i < E; ++i) S[j][i] = ix_wire(C[j][i], (const TIO*)nullptr);
      }
    }
    if (nt == T) {
      // Skewed by half a token: an iteration joins the two trees that are pending (k dot of this token, q dot of the one
      // before, so that neither waits alone for its lane exchanges), updates the state, and issues the dots of its own q
      // and the next token's k. k is loaded two tokens ahead, q one; the scheduling barrier keeps those loads at the top
      // of the iteration, a whole one in front of their use (left alone, the compiler sinks them to it).
      float kb[3][E], qb[2][E], vb3[3][RPL], kp[RPL], qp[RPL], cp[RPL], keep[RPL];
      auto put = [&](int tt, int j, float ov) __attribute__((always_inline)) {
        if ((tt % L) == 0) keep[j] = ov;
        else keep[j] = sub == tt % L ? ov : keep[j];
        if (tt % L == L - 1 || tt == T - 1) { if (T - tt / L * L >= L || sub < T % L) of[b][tt / L * L + sub][j * RW + r] = keep[j]; }
      };
      // The output of the token before is put away ahead of the update, or after it where a wave has its SIMD nearly to itself
      // (LONE) or one bf16 state. us after / ahead, boundary form of fp32, K = V = 128, 32 heads: 32 x 200 tokens 759 / 744, 64 x
      // 64 484 / 469; one state in bf16, 2000 tokens beside seven times 16 446 / 453.
      constexpr bool PUT_FIRST = !LONE && (CPR || sizeof(TIO) == 4);
      float2 gb[3];
      auto load_k = [&](int tt) __attribute__((always_inline)) {
        load_x(&kq[b][0][tt][0], kb[tt % 3]);
        gb[tt % 3] = eb[b][tt];
#pragma unroll
        for (int j = 0; j < RPL; ++j) vb3[tt % 3][j] = vf[b][tt][j * RW + r];
      };
      auto load_q = [&](int tt) __attribute__((always_inline)) { load_x(&kq[b][1][tt][0], qb[tt % 2]); };
      auto decay_dot = [&](int tt) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < RPL; ++j) {
#pragma unroll
          for (int i = 0; i < E; ++i) S[j][i] = S[j][i] * gb[tt % 3].x;
          kp[j] = ix_dot_slice(S[j], kb[tt % 3]);
          if constexpr (CPR) {
#pragma unroll
            for (int i = 0; i < E; ++i) C[j][i] = C[j][i] * gb[tt % 3].x;
            cp[j] = ix_dot_slice(C[j], kb[tt % 3]);
          }
        }
      };
      load_k(0);
      load_k(1);
      load_q(0);
      decay_dot(0);
#pragma unroll
      for (int tt = 0; tt < T; ++tt) {
        if (tt + 2 < T) load_k(tt + 2);
        if (tt + 1 < T) load_q(tt + 1);
        __builtin_amdgcn_sched_barrier(0);
        float ov[RPL], kv[RPL], cv[RPL];
#pragma unroll
        for (int j = 0; j < RPL; ++j) {
          kv[j] = ix_lane_tree<L>(kp[j]);
          if constexpr (CPR) cv[j] = ix_lane_tree<L>(cp[j]);
          if (tt > 0) ov[j] = ix_lane_tree<L>(qp[j]);
        }
#pragma unroll
        for (int j = 0; j < RPL; ++j) {
          if (PUT_FIRST && tt > 0) put(tt - 1, j, ov[j]);
          const float d = (vb3[tt % 3][j] - kv[j]) * gb[tt % 3].y;
#pragma unroll
          for (int i = 0; i < E; ++i) S[j][i] = __builtin_fmaf(d, kb[tt % 3][i], S[j][i]);
          qp[j] = ix_dot_slice(S[j], qb[tt % 2]);
          if constexpr (CPR) {
            const float dc = (vb3[tt % 3][j] - cv[j]) * gb[tt % 3].y;
#pragma unroll
            for (int i = 0; i < E; ++i) C[j][i] = __builtin_fmaf(dc, kb[tt % 3][i], C[j][i]);
          }
        }
        if (!PUT_FIRST && tt > 0) {
#pragma unroll
          for (int j = 0; j < RPL; ++j) put(tt - 1, j, ov[j]);
        }
        if (tt + 1 < T) decay_dot(tt + 1);
      }
#pragma unroll
      for (int j = 0; j < RPL; ++j) put(T - 1, j, ix_lane_tree<L>(qp[j]));
    } else {
      // All lanes of a row have its output and store it, but where one lane's store leaves the faster code (boundary form in
      // bf16, K = V = 128, 32 heads, 32 x 200 tokens 777 / 747 us; without a second state in the LONE form 157 / 161).
      constexpr bool ONE_STORES = CPR && !LONE && sizeof(TIO) == 2;
      for (int tt = 0; tt < nt; ++tt) {
        float kk[E], qs[E];
        load_x(&kq[b][0][tt][0], kk);
        load_x(&kq[b][1][tt][0], qs);
        const float2 gb = eb[b][tt];
#pragma unroll
        for (int j = 0; j < RPL; ++j) {
          const float vv = vf[b][tt][j * RW + r];
          auto advance = [&](float (&X)[E]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < E; ++i) X[i] = X[i] * gb.x;
            const float d = (vv - ix_lane_tree<L>(ix_dot_slice(X, kk))) * gb.y;
#pragma unroll
            for (int i = 0; i < E; ++i) X[i] = __builtin_fmaf(d, kk[i], X[i]);
          };
          if constexpr (CPR) advance(C[j]);
          advance(S[j]);
          const float ov = ix_lane_tree<L>(ix_dot_slice(S[j], qs));
          if (!ONE_STORES || sub == 0) of[b][tt][j * RW + r] = ov;
        }
      }
    }
    if constexpr (!LONE) {
      if (it + 1 < tiles) commit(b ^ 1);
    }
    __syncthreads();
  }
  if constexpr (!LONE) emit((tiles - 1) * T, len - (tiles - 1) * T, (tiles - 1) & 1);
  if (state && !CPR) {
#pragma unroll
    for (int j = 0; j < RPL; ++j) {
      float* sp = state + (((long)row0 * HV + hv) * V + vb * R + r + j * RW) * K + kbase;
      if constexpr (E == 8) {
        *reinterpret_cast<float4*>(sp) = make_float4(S[j][0], S[j][1], S[j][2], S[j][3]);
        *reinterpret_cast<float4*>(sp + 4) = make_float4(S[j][4], S[j][5], S[j][6], S[j][7]);
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) sp[i * 2] = S[j][i];
      }
    }
  }
}

// ---- the walk with four lanes per row (K = 128) ---------------------------------------------------------------
// k_gdn_walk's staging (two tiles of 16 tokens, one barrier per tile) around k_gdn_scan_quads' token with ONE row per lane: a
// wave has sixteen rows, a workgroup 64. CPR: the lane's second state is the fp32 chain beside the running state, and its row's
// reads of k serve both. Outputs stay in registers for four tokens, so that those tokens' reads of LDS may pass one another.
// Bound by vector issue with several waves per SIMD: 128 instructions per token for sixteen rows, 202 in the boundary form.
// Tried: the next token's reads and dot products between a token's update and its output (168 registers no longer hold it;
// with two waves per SIMD 64 x 1000 tokens of the boundary form 5466 -> 6221 us); one element of k and q per lane, broadcast on
// the operand path of the multiply-adds, instead of the LDS reads (those multiply-adds do not run at the full rate: 6646); a
// higher wave priority for the longer sequences (nothing).
template <typename TIO, bool CPR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void k_gdn_walk_quads(const TIO* __restrict__ q, const TIO* __restrict__ k, const TIO* __restrict__ v,
                      const float* __restrict__ g, const TIO* __restrict__ beta, TIO* __restrict__ o,
                      float* __restrict__ state, const int* __restrict__ cu, const int* __restrict__ sidx, long q_pitch,
                      long k_pitch, long v_pitch, int N, int H, int HV, int V, float scale, int chunk) {
  constexpr int K = 128, T = 16, R = 64, J = CPR ? 2 : 1;
  constexpr int Q = IX_QUAD_KP, VAT = 2 * IX_QUAD_KP, OAT = VAT + R, EAT = OAT + R, REC = EAT + 4;
  constexpr int VC = T * R / 256;
  __shared__ __align__(16) float rec[2][T * REC];  // a token: k, q * scale [IX_QUAD_KP each], v [R], o [R], exp(g), beta
  static_assert(sizeof(rec) >= (IX_GDN_SORT_MAX + 1) * sizeof(int), "the ranking uses the staging buffer");

  const int VB = V / R;
  const int per_seq = HV * VB;
  const int tid = threadIdx.x;
  int n, w;
  {
    const unsigned bid = blockIdx.x;
    if ((per_seq & 7) == 0) {  // hardware deals consecutive ids to the XCDs round-robin
      const unsigned per8 = (unsigned)per_seq >> 3;
      // Every second round of 32 workgroups of an XCD, one per CU, runs the other way: the CU with the longest sequence gets the
      // shortest of the next round.
      unsigned p = bid >> 3;
      const unsigned all = (unsigned)N * per8, first = p & ~31u;
      if (first & 32u) p = first + min(31u, all - 1 - first) - (p & 31u);
      n = (int)(p / per8);
      w = (int)((bid & 7u) * per8 + p % per8);
    } else {
      n = (int)(bid / (unsigned)per_seq);
      w = (int)(bid % (unsigned)per_seq);
    }
  }
  n = ix_gdn_nth_longest(cu, N, n, reinterpret_cast<int*>(&rec[0][0]));
  const int vb = w % VB;
  const int hv = w / VB;
  const int h = hv / (HV / H);
  const int t_begin = cu[n];
  const int len = cu[n + 1] - t_begin;
  if (len <= 0) return;
  const int row0 = sidx ? sidx[n] : 1;
  TIO* ob = o + (long)hv * V + vb * R;
  if (row0 <= 0) {  // null lane: no state, outputs defined as zero
    for (int i = tid; i < len * R; i += 256) ix_st(ob + (long)(t_begin + i / R) * HV * V + i % R, 0.0f);
    return;
  }
  const int tiles = (len + T - 1) / T;

  // staging: a thread has one group of eight of k and of q, VC values of v
  const int gt = tid >> 4, gk = (tid & 15) * 8;
  IxRaw8<TIO> rk, rq;
  TIO rv[VC], rb = 0;
  float rg = 0.0f;
  auto fetch = [&](int t0) __attribute__((always_inline)) {  // tokens past the end read the last one's values, unused
    const long tok = t_begin + min(t0 + gt, len - 1);
    rk.load(k + tok * k_pitch + h * K + gk);
    rq.load(q + tok * q_pitch + h * K + gk);
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      const int i = tid + 256 * c;
      rv[c] = v[(t_begin + min(t0 + i / R, len - 1)) * v_pitch + (long)hv * V + vb * R + i % R];
    }
    if (tid < T) {
      const long src = (t_begin + (long)min(t0 + tid, len - 1)) * HV + hv;
      rg = g[src];
      rb = beta[src];
    }
  };
  auto commit = [&](int b) __attribute__((always_inline)) {
    float x[8], y[8];
    rk.widen(x);
    rq.widen(y);
    float* d = &rec[b][gt * REC + ix_quad_at(gk)];
    *reinterpret_cast<float4*>(d) = make_float4(x[0], x[1], x[2], x[3]);
    *reinterpret_cast<float4*>(d + 4) = make_float4(x[4], x[5], x[6], x[7]);
    *reinterpret_cast<float4*>(d + Q) = make_float4(y[0] * scale, y[1] * scale, y[2] * scale, y[3] * scale);
    *reinterpret_cast<float4*>(d + Q + 4) = make_float4(y[4] * scale, y[5] * scale, y[6] * scale, y[7] * scale);
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      const int i = tid + 256 * c;
      rec[b][i / R * REC + VAT + i % R] = ix_ld(&rv[c]);
    }
    if (tid < T) *reinterpret_cast<float2*>(&rec[b][tid * REC + EAT]) = make_float2(ix_exp(rg), ix_ld(&rb));
  };
  auto emit = [&](int t0, int nt, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      const int i = tid + 256 * c;
      if (i < nt * R) ix_st(ob + (long)(t_begin + t0 + i / R) * HV * V + i % R, rec[b][i / R * REC + OAT + i % R]);
    }
  };

  const int lane = tid & 63, wave = tid >> 6;
  const int grp = lane >> 4;
  const int r = wave * 16 + (lane & 15);
  // S[0]: the state that makes the outputs, S[1]: the chain; S[j][c][i]: k = 32 grp + 16 c + i
  ix_f32x16 S[J][2];
  float* srow = state + (((long)row0 * HV + hv) * V + vb * R + r) * K + 32 * grp;
#pragma unroll
  for (int j = 0; j < J; ++j) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float4 a = state ? *reinterpret_cast<const float4*>(srow + 4 * c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      ix_f32x16& d = S[j][c >> 2];
      const int i = 4 * (c & 3);
      d[i] = a.x; d[i + 1] = a.y; d[i + 2] = a.z; d[i + 3] = a.w;
    }
  }
  // the element of k that this lane hands to the update's first instruction (the second one's: 16 further)
  const int ka = 36 * ((lane & 15) >> 2) + 4 * grp + (lane & 3);

  fetch(0);
  commit(0);
  __syncthreads();
  for (int it = 0; it < tiles; ++it) {
    const int b = it & 1, t0 = it * T;
    const int nt = min(T, len - t0);
    if (it + 1 < tiles) fetch(t0 + T);
    if (it > 0) emit(t0 - T, T, b ^ 1);
    if constexpr (CPR) {
      if (t0 % chunk == 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 16; ++i) S[0][c][i] = ix_wire(S[1][c][i], (const TIO*)nullptr);
      }
    }
    auto token = [&](int tt) __attribute__((always_inline)) {
      const float* at = &rec[b][tt * REC];
      const float eg = at[EAT], bt = at[EAT + 1], vv = at[VAT + r];
      float x[32];  // this lane group's elements of k, later of q
      ix_quad_load(at, grp, x);
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 16; ++i) S[j][c][i] = S[j][c][i] * eg;
      // CPR: groups 0 and 2 go on with the running state, 1 and 3 with the chain
      const float p0 = ix_quad_dot(S[0], x);
      const float p1 = CPR ? ix_quad_dot(S[J - 1], x) : p0;
      const float d = (vv - ix_add_groups2(p0, p1)) * bt;
      float dj[2] = {d, d};
      if constexpr (CPR) {  // each to all four groups
        const auto dd = __builtin_amdgcn_permlane16_swap(__float_as_uint(d), __float_as_uint(d), false, false);
        dj[0] = __uint_as_float(dd[0]);
        dj[1] = __uint_as_float(dd[1]);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float ke = at[ka + 16 * c];
#pragma unroll
        for (int j = 0; j < J; ++j) S[j][c] = __builtin_amdgcn_mfma_f32_16x16x1f32(ke, dj[j], S[j][c], 0, 0, 0);
      }
      ix_quad_load(at + Q, grp, x);
      const float p = ix_quad_dot(S[0], x);
      return ix_add_groups2(p, p);
    };
    int tt = 0;
    for (; tt + 4 <= nt; tt += 4) {
      float ov[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) ov[u] = token(tt + u);
#pragma unroll
      for (int u = 0; u < 4; ++u) rec[b][(tt + u) * REC + OAT + r] = ov[u];  // every group of the row has it
    }
    for (; tt < nt; ++tt) rec[b][tt * REC + OAT + r] = token(tt);
    if (it + 1 < tiles) commit(b ^ 1);
    __syncthreads();
  }
  emit((tiles - 1) * T, len - (tiles - 1) * T, (tiles - 1) & 1);
  if (state && !CPR) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const ix_f32x16& a = S[0][c >> 2];
      const int i = 4 * (c & 3);
      *reinterpret_cast<float4*>(srow + 4 * c) = make_float4(a[i], a[i + 1], a[i + 2], a[i + 3]);
    }
  }
}

// q and k rows that can be fetched 8 elements at a time: every row start on a 16-byte (bf16) or 32-byte (fp32) boundary
template <typename TIO>
static bool ix_gdn_vec_qk(const void* q, const void* k, long q_pitch, long k_pitch) {
  return q_pitch % 8 == 0 && k_pitch % 8 == 0 && ix_aligned(q, 8 * sizeof(TIO)) && ix_aligned(k, 8 * sizeof(TIO));
}

template <int K, int E, typename TIO, bool CPR>
static int ix_gdn_walk_launch(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                              float* state, const int* cu, const int* sidx, long q_pitch, long k_pitch, long v_pitch,
                              long N, int H, int HV, int V, float scale, int chunk, int rpl, bool lone, hipStream_t st) {
  constexpr int RW = 256 / (K / E);  // split slices come in the lone form only
  if (V % RW != 0 || !ix_gdn_vec_qk<TIO>(q, k, q_pitch, k_pitch)) return IX_DECLINED;
  if (rpl == 2 && V % (2 * RW) != 0) rpl = 1;
  const long grid = N * HV * (V / (RW * rpl));
  if (grid > 0x7fffffffL) return IX_DECLINED;
#define IX_WALK(RPL_, LONE_)                                                                                           \
  hipLaunchKernelGGL((k_gdn_walk<K, E, RPL_, TIO, CPR, LONE_>), dim3((unsigned)grid), dim3(LONE_ ? 320 : 256), 0, st, \
                     (const TIO*)q, (const TIO*)k, (const TIO*)v, g, (const TIO*)beta, (TIO*)o, state, cu, sidx,        \
                     q_pitch, k_pitch, v_pitch, (int)N, H, HV, V, scale, chunk)
  if constexpr (E == 4) {
    IX_WALK(1, true);
  } else {
    if (rpl == 2) IX_WALK(2, false);
    else if (lone) IX_WALK(1, true);
    else IX_WALK(1, false);
  }
#undef IX_WALK
  return ix_launch_status();
}

static size_t ix_gdn_lds_bytes(int K, int R, int TT) {
  return (size_t)TT * (2 * K + 2 * R + 3) * sizeof(float);
}

template <int KS, int RPL, typename TIO>
static int ix_gdn_scan_launch_rpl(const void* q, const void* k, const void* v, const float* g, const void* beta,
                                  void* o, float* state, const int* cu, const int* sidx, long sidx_stride,
                                  long q_pitch, long k_pitch, long v_pitch, long N, int H, int HV, int V, float scale,
                                  int TT, hipStream_t st) {
  constexpr int R = (256 / KS) * RPL;
  if (V % R != 0) return IX_DECLINED;
  const long grid = N * HV * (V / R);
  if (grid > 0x7fffffffL) return IX_DECLINED;
  const size_t lds = ix_gdn_lds_bytes(KS * 8, R, TT);
  auto kern = k_gdn_scan<KS, RPL, TIO>;
  if (lds > 48 * 1024) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return IX_ERR_LAUNCH;
  }
  // workgroup order = state order in the pool, walked in 8 XCD runs (a decode step streams the pool once:
  // 0.214 -> 0.210 ms at 256 sequences)
  const unsigned xcd_total = (unsigned)grid;
  if (xcd_total > 0x7ffffff0u) return IX_DECLINED;
  hipLaunchKernelGGL(kern, dim3(ix_xcd_run_grid(xcd_total)), dim3(256), lds, st,
                     (const TIO*)q, (const TIO*)k, (const TIO*)v, g, (const TIO*)beta, (TIO*)o, state, cu, sidx,
                     sidx_stride, q_pitch, k_pitch, v_pitch, H, HV, V, scale, TT, xcd_total);
  return ix_launch_status();
}

// Rows per lane group: a staging choice like the time tile (bits 8.. of time_tile force it). More rows per
// workgroup share each k/q fetch and interleave independent chains, but leave fewer workgroups.
template <int KS, typename TIO>
static int ix_gdn_scan_launch(const void* q, const void* k, const void* v, const float* g, const void* beta,
                              void* o, float* state, const int* cu, const int* sidx, long sidx_stride,
                              long q_pitch, long k_pitch, long v_pitch, long N, int H, int HV, int V, float scale,
                              int TT, int rpl, hipStream_t st) {
  constexpr int RW = 256 / KS;
  if (V % RW != 0) return IX_DECLINED;
  const long groups = N * HV * (V / RW);  // workgroups at one row per lane group
  if (rpl <= 0) rpl = (V % (RW * 2) == 0 && groups >= 2 * 1024) ? 2 : 1;  // measured: 4 rows gain nothing over 2
  while (rpl > 1 && V % (RW * rpl) != 0) rpl >>= 1;
#define IX_RPL_CASE(R_)                                                                                          \
  case R_:                                                                                                       \
    return ix_gdn_scan_launch_rpl<KS, R_, TIO>(q, k, v, g, beta, o, state, cu, sidx, sidx_stride, q_pitch, k_pitch, \
                                               v_pitch, N, H, HV, V, scale, TT, st);
  switch (rpl) {
    IX_RPL_CASE(1)
    IX_RPL_CASE(2)
    IX_RPL_CASE(4)
    default:
      return IX_ERR_ARG;
  }
#undef IX_RPL_CASE
}

// Which layout runs whole sequences at K = 128: 0 the sixteen-lane walk, IX_GDN_FOUR_ONE four lanes per row with one row per lane
// (k_gdn_walk_quads), IX_GDN_FOUR_TWO with two (k_gdn_scan_quads); the values are time_tile's layout codes. Four lanes issue 8
// (two rows per lane 7.5) vector instructions per row and token where the walk issues 11, in the boundary form 13 where it
// issues 18. But a token takes a lone wave 0.42 us (two rows 0.9, boundary form 0.58) where the walk's takes 0.12 to 0.22, so
// the longest sequence decides: four lanes pay where enough of the others run beside it to its end. `even`: the tokens as so many
// sequences of the longest one's length, in workgroups of 64 rows. us walk / one row / two rows, 32 heads, V = 128 (64
// workgroups a sequence), bf16, `even` in brackets:
//   1 x 8000 + 15 x 100 tokens (76) 1782 / 3335 / 6758     1 x 4096 + 31 x 64 (95) 912 / 1714 / 3401
//   4 x 2000 + 12 x 200 (332) 779 / 870 / 1755             6 x 2000 + 10 x 200 (448) 1023 / 1033 / 1814
//   16 of 60..1410 (533) 874 / 706 / 1295                  1 x 3000 + 47 x 500 (565) 1920 / 1565 / 2931
//   8 x 2000 + 40 x 100 (640) 1453 / 1169 / 1849           16 x 1000 (1024) 1148 / 1000 / 1061
//   48 of 60..1470 (1598) 2491 / 2085 / 2169               24 x 1000 + 24 x 100 (1689) 1791 / 1479 / 1401
//   48 x 1000 (3072) 3327 / 2810 / 2720                    12 of 60..1380 (768 workgroups) 595 / 628 / 1165
// Two rows per lane also take the gated norm along, which is worth more than the 4 % that they lose at 1598. Short sequences,
// where a launch's start counts: 16 x 24 41 / 42, 16 x 48 64 / 64, 32 x 24 72 / 71, 32 x 32 88 / 80, 48 x 16 77 / 78 / 83, 63 x 20
// 123 / 113 / 127, 63 x 24 141 / 127 / 130.
// Boundary form, walk / one row: 1 x 4096 + 31 x 64 (95) 1350 / 2361, 2 x 2000 + 14 x 200 (217) 803 / 1175, 4 x 2000 + 12 x 200
// (332) 1202 / 1190, ten of 120..1500 (345) 942 / 915, 8 x 1000 + 2 x 100 (524) 994 / 767, 200 x 9 411 / 262, 64 x 1000 7274 /
// 5414; nine of 120..1500 (576 workgroups) were 1008 / 1000; fp32: 4 x 2000 + 28 x 200 (435) 1650 / 1488, 16 of 60..1500 (532)
// 1423 / 1200, nine of 120..1500 1025 / 1119.
// Where the host does not know the lengths (longest <= 0) only IX_GDN_QUAD_MANY workgroups of 128 rows leave the walk: 64 x 1000
// tokens 4413 / 3845 / 3495.
#define IX_GDN_FOUR_TWO 16
#define IX_GDN_FOUR_ONE 19
#define IX_GDN_QUAD_MANY 2048
#define IX_GDN_QUAD_MIN 1536  // the same with known lengths, and for a state-only pass
static int ix_gdn_layout_for(long N, long HV, long V, long tokens, long longest, bool bf16, bool boundary) {
  const long wgs = N * HV * (V / 64), pairs = V % 128 == 0 ? wgs / 2 : 0;
  if (longest <= 0) return !boundary && pairs >= IX_GDN_QUAD_MANY ? IX_GDN_FOUR_TWO : 0;
  if (V % 64 != 0) return 0;
  const long even = tokens * HV * (V / 64) / longest;
  if (boundary) return wgs >= (bf16 ? 640 : 1024) && even >= (bf16 ? 320 : 448) ? IX_GDN_FOUR_ONE : 0;
  if (even >= 1536 && (pairs >= IX_GDN_QUAD_MANY || (pairs >= IX_GDN_QUAD_MIN && tokens >= 24 * N))) return IX_GDN_FOUR_TWO;
  return wgs >= 1024 && even >= 448 && tokens >= 20 * N && tokens * HV * (V / 64) >= 49152 ? IX_GDN_FOUR_ONE : 0;
}

// chunk > 0: the boundary form. rpl: state rows per lane group of sixteen, 3 = four lanes per row, 0 = one or two by the rule below.
static int ix_gdn_walk(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                       int io_dtype, float* state, const int* cu, const int* sidx, long q_pitch, long k_pitch, long v_pitch,
                       long N, int H, int HV, long K, int V, float scale, int chunk, int rpl, hipStream_t st) {
  // Two rows per lane group share the LDS reads of k and q and give a wave two chains to interleave, one leaves twice the
  // waves. Measured at HV = 32, V = K = 128, us one / two rows: one sequence of 8192 tokens 1129 / 1823, five of 33..1203
  // 247 / 307, nine of 120..1500 608 / 591, 16 x 1000 1266 / 1180; K = V = 64, HV = 16
  // and 32: 8 x 500 72 / 110, 32 x 500 329 / 323. The line: eight waves per SIMD at one row.
  // Fewer workgroups: a wave of their own stages the tiles (LONE) up to two of them per CU; with more, its registers and its
  // share of the issue are missed. us without / with it: one sequence of 8192 tokens 1147 / 988, 2 x 3000 544 / 501, 3 x 2000
  // 484 / 522; K = V = 64, HV = 32, 8 x 512 92 / 86, 16 x 512 156 / 210. Two of them per CU are ten waves, which need 128
  // registers at most: the fp32 forms of K >= 128 (138 and 146, the raw tile in the staging wave) stop at one (16 heads, K =
  // 128, 3 x 1000 tokens 185 / 240, 4 x 700 132 / 173; K = 256, 8 heads 242 / 305). And a slice split over two lanes (E = 4)
  // while one such workgroup per CU, two at K <= 64, is all there is (at K = 128 a row is then 32 lanes and its tree has a
  // level across the halves of 16). us whole / split: 2000 tokens of 16 heads at K = 128 245 / 206, of 32 heads (two per CU)
  // 66 / 75 per 500; K = 64, 2 x 256 of 4 heads 33 / 24, 8 x 512 of 16 heads 66 / 63, of 32 heads 86 / 107.
  const long quad_wgs = N * HV * (V / 64);
  const bool vec_qk = io_dtype == IX_DT_BF16 ? ix_gdn_vec_qk<bf16_t>(q, k, q_pitch, k_pitch)
                                             : ix_gdn_vec_qk<float>(q, k, q_pitch, k_pitch);
  if (rpl == 3) {
    if (K != 128 || V % 64 != 0 || quad_wgs > 0x7fffffffL || !vec_qk) return IX_DECLINED;
#define IX_WALK_QUADS(TIO, CPR_)                                                                                     \
  hipLaunchKernelGGL((k_gdn_walk_quads<TIO, CPR_>), dim3((unsigned)quad_wgs), dim3(256), 0, st, (const TIO*)q, (const TIO*)k, \
                     (const TIO*)v, g, (const TIO*)beta, (TIO*)o, state, cu, sidx, q_pitch, k_pitch, v_pitch, (int)N, H, \
                     HV, V, scale, chunk)
    if (io_dtype == IX_DT_BF16) {
      if (chunk > 0) { IX_WALK_QUADS(bf16_t, true); } else { IX_WALK_QUADS(bf16_t, false); }
    } else {
      if (chunk > 0) { IX_WALK_QUADS(float, true); } else { IX_WALK_QUADS(float, false); }
    }
#undef IX_WALK_QUADS
    return ix_launch_status();
  }
  const long lanes = N * HV * V * (K / 8);  // threads at one row per lane group, whole slices
  const bool auto_shape = rpl <= 0;
  if (auto_shape) rpl = lanes >= 8L * 1024 * 64 ? 2 : 1;
  const bool lone = auto_shape && lanes <= (io_dtype == IX_DT_F32 && K >= 128 ? 1L : 2L) * 256 * 256;
  const bool split = auto_shape && K <= 128 && 2 * lanes <= (K == 128 ? 256L : 512L) * 256 &&
                     V % (2048 / K) == 0;  // what whole slices decline stays declined
#define IX_WALK_ARGS(CHUNK_) \
  q, k, v, g, beta, o, state, cu, sidx, q_pitch, k_pitch, v_pitch, N, H, HV, V, scale, CHUNK_, rpl, lone, st
#define IX_WALK_CASE(KV, EV)                                                                            \
  if (K == KV && split == (EV == 4)) {                                                                  \
    if (io_dtype == IX_DT_BF16)                                                                         \
      return chunk > 0 ? ix_gdn_walk_launch<KV, EV, bf16_t, true>(IX_WALK_ARGS(chunk))                  \
                       : ix_gdn_walk_launch<KV, EV, bf16_t, false>(IX_WALK_ARGS(0));                    \
    return chunk > 0 ? ix_gdn_walk_launch<KV, EV, float, true>(IX_WALK_ARGS(chunk))                     \
                     : ix_gdn_walk_launch<KV, EV, float, false>(IX_WALK_ARGS(0));                       \
  }
  IX_WALK_CASE(32, 4)
  IX_WALK_CASE(64, 4)
  IX_WALK_CASE(128, 4)
  IX_WALK_CASE(32, 8)
  IX_WALK_CASE(64, 8)
  IX_WALK_CASE(128, 8)
  IX_WALK_CASE(256, 8)
#undef IX_WALK_CASE
#undef IX_WALK_ARGS
  return IX_DECLINED;
}

static int ix_gdn_quads(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o, int io_dtype,
                        long q_pitch, long k_pitch, long v_pitch, float* state, const int* cu, const int* sidx, long N,
                        int H, int HV, int V, float scale, int TT, const bf16_t* gate, long gate_stride_t,
                        const bf16_t* norm_w, float norm_eps, int zero_centered, hipStream_t st) {
  const long grid = N * HV * (V / 128);
  if (grid > 0x7fffffffL) return IX_DECLINED;
  size_t lds = (size_t)TT * (2 * IX_QUAD_KP + 2 * 128 + 4) * sizeof(float);
  if (lds < (IX_GDN_SORT_MAX + 1) * sizeof(int)) lds = (IX_GDN_SORT_MAX + 1) * sizeof(int);
  if (io_dtype == IX_DT_BF16)
    hipLaunchKernelGGL((k_gdn_scan_quads<bf16_t>), dim3((unsigned)grid), dim3(256), lds, st, (const bf16_t*)q,
                       (const bf16_t*)k, (const bf16_t*)v, g, (const bf16_t*)beta, (bf16_t*)o, state, cu, sidx, q_pitch,
                       k_pitch, v_pitch, (int)N, H, HV, V, scale, TT, gate, gate_stride_t, norm_w, norm_eps, zero_centered);
  else
    hipLaunchKernelGGL((k_gdn_scan_quads<float>), dim3((unsigned)grid), dim3(256), lds, st, (const float*)q,
                       (const float*)k, (const float*)v, g, (const float*)beta, (float*)o, state, cu, sidx, q_pitch, k_pitch,
                       v_pitch, (int)N, H, HV, V, scale, TT, (const bf16_t*)nullptr, 0L, (const bf16_t*)nullptr, 0.0f, 0);
  return ix_launch_status();
}

static int ix_gdn_scan_impl(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                            int io_dtype, long q_pitch, long k_pitch, long v_pitch, float* state_pool,
                            const int* cu_seqlens, const int* state_indices, long state_indices_stride, long N,
                            long H, long HV, long K, long V, float scale, int time_tile, const bf16_t* gate,
                            long gate_stride_t, const bf16_t* norm_w, float norm_eps, int zero_centered, long tokens,
                            long longest, void* stream) {
  if (!q || !k || !v || !g || !beta || !state_pool || !cu_seqlens || !state_indices) return IX_ERR_ARG;
  if (N < 0 || H <= 0 || HV <= 0 || K <= 0 || V <= 0 || HV % H != 0 || state_indices_stride < 0) return IX_ERR_ARG;
  if (q_pitch < H * K || k_pitch < H * K || v_pitch < HV * V) return IX_ERR_ARG;
  if (io_dtype != IX_DT_F32 && io_dtype != IX_DT_BF16) return IX_DECLINED;
  if (N == 0) return IX_OK;
  if (!ix_aligned(state_pool, 16)) return IX_DECLINED;
  const int rpl = time_tile > 0 ? (time_tile >> 8) : 0;
  // default time tile: short tiles keep more workgroups resident when there are many, long tiles
  // amortise the staging when there are few
  int TT = time_tile <= 0 ? 0 : (time_tile & 0xff);
  if (TT <= 0) TT = (N * HV * (V / 16) >= 4096) ? 16 : 64;
  if (TT > 64) TT = 64;
  hipStream_t st = (hipStream_t)stream;
  // Four lanes per row: compact state form, K = 128, where ix_gdn_layout_for says so (or forced by code 16 or 19 in bits 8.. of
  // time_tile). A time tile of 1 says one token per sequence (a decode step): that is a pure stream of the state, which
  // the 16-lane layout does with more waves in flight. A state-only pass (the boundary pass of a decode step: equal lengths, most
  // rows null lanes) has k_gdn_scan to compare with: 63 rows of 64 tokens, us k_gdn_scan / four lanes with no row live 8.5 / 10.2,
  // one 46 / 52, four 154 / 54, all 321 / 235.
  const bool compact = state_indices_stride == 0 && K == 128;
  int layout = 0;
  if (compact && rpl == 0 && (time_tile & 0xff) != 1) {
    layout = ix_gdn_layout_for(N, HV, V, tokens, longest, io_dtype == IX_DT_BF16, false);
    if (!o && V % 128 == 0 && N * HV * (V / 128) >= IX_GDN_QUAD_MIN) layout = IX_GDN_FOUR_TWO;
  }
  if (compact && V % 128 == 0 && (rpl == 16 || layout == IX_GDN_FOUR_TWO))
    return ix_gdn_quads(q, k, v, g, beta, o, io_dtype, q_pitch, k_pitch, v_pitch, state_pool, cu_seqlens, state_indices, N,
                        (int)H, (int)HV, (int)V, scale, time_tile > 0 && (time_tile & 0xff) > 0 ? TT : 16, gate,
                        gate_stride_t, norm_w, norm_eps, zero_centered, st);
  if (gate) return IX_DECLINED;       // the norm rides on two rows per lane only
  if (rpl == 16) return IX_DECLINED;  // that layout was asked for and does not apply
  // Sequences of more than one token in the compact form: the walk (codes 17 and 18 force it with one and two rows per
  // lane group, 19 with four lanes per row). k_gdn_scan below keeps the decode step, the per-token index map, the state-only
  // pass and the operands whose rows are not aligned.
  if (state_indices_stride == 0 && o && (time_tile <= 0 || (rpl >= 17 && rpl <= 19))) {
    const int form = rpl >= 17 ? rpl - 16 : (layout == IX_GDN_FOUR_ONE ? 3 : 0);
    const int rc = ix_gdn_walk(q, k, v, g, beta, o, io_dtype, state_pool, cu_seqlens, state_indices, q_pitch, k_pitch,
                               v_pitch, N, (int)H, (int)HV, K, (int)V, scale, 0, form, st);
    if (rc != IX_DECLINED) return rc;
  }
  if (rpl >= 17) return IX_DECLINED;
#define IX_SCAN_CASE(KSV)                                                                                         \
  if (K == KSV * 8) {                                                                                             \
    if (io_dtype == IX_DT_BF16)                                                                                   \
      return ix_gdn_scan_launch<KSV, bf16_t>(q, k, v, g, beta, o, state_pool, cu_seqlens, state_indices,         \
                                             state_indices_stride, q_pitch, k_pitch, v_pitch, N, (int)H,         \
                                             (int)HV, (int)V, scale, TT, rpl, st);                               \
    return ix_gdn_scan_launch<KSV, float>(q, k, v, g, beta, o, state_pool, cu_seqlens, state_indices,            \
                                          state_indices_stride, q_pitch, k_pitch, v_pitch, N, (int)H, (int)HV,   \
                                          (int)V, scale, TT, rpl, st);                                           \
  }
  IX_SCAN_CASE(4)
  IX_SCAN_CASE(8)
  IX_SCAN_CASE(16)
  IX_SCAN_CASE(32)
#undef IX_SCAN_CASE
  return IX_DECLINED;
}

extern "C" int ix_gdn_scan(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                           int io_dtype, long q_pitch, long k_pitch, long v_pitch, float* state_pool,
                           const int* cu_seqlens, const int* state_indices, long state_indices_stride, long N,
                           long H, long HV, long K, long V, float scale, int time_tile, void* stream) {
  return ix_gdn_scan_impl(q, k, v, g, beta, o, io_dtype, q_pitch, k_pitch, v_pitch, state_pool, cu_seqlens, state_indices,
                          state_indices_stride, N, H, HV, K, V, scale, time_tile, nullptr, 0, nullptr, 0.0f, 0, 0, 0, stream);
}

// The gated output norm (ix_gated_out_norm with N = V) in the scan's launch: o receives bf16(norm(o_scan) * silu(gate)) instead of
// o_scan -- the bits of the two calls. What its operands have to be, whatever the layout rule says.
static bool ix_gdn_norm_fits(const void* o, int io_dtype, long K, long V, const void* gate, long gate_stride_t, const void* w) {
  return io_dtype == IX_DT_BF16 && K == 128 && V == 128 && gate_stride_t % 8 == 0 && ix_aligned(gate, 16) && ix_aligned(w, 16) &&
         ix_aligned(o, 16);
}

// Declines (IX_DECLINED) before anything is launched or the state is touched where two rows per lane do not run.
extern "C" int ix_gdn_scan_gated_norm(const void* q, const void* k, const void* v, const float* g, const void* beta,
                                      void* o, long q_pitch, long k_pitch, long v_pitch, float* state_pool,
                                      const int* cu_seqlens, const int* state_indices, long N, long H, long HV, long K,
                                      long V, float scale, int time_tile, const void* gate, long gate_stride_t,
                                      const void* norm_weight, float norm_eps, int zero_centered, void* stream) {
  if (!o || !gate || !norm_weight || gate_stride_t < HV * V) return IX_ERR_ARG;
  if (!ix_gdn_norm_fits(o, IX_DT_BF16, K, V, gate, gate_stride_t, norm_weight) || (time_tile & 0xff) == 1 ||
      (time_tile >> 8) != 0 || N * HV < IX_GDN_QUAD_MANY)
    return IX_DECLINED;
  return ix_gdn_scan_impl(q, k, v, g, beta, o, IX_DT_BF16, q_pitch, k_pitch, v_pitch, state_pool, cu_seqlens,
                          state_indices, 0, N, H, HV, K, V, scale, time_tile, (const bf16_t*)gate, gate_stride_t,
                          (const bf16_t*)norm_weight, norm_eps, zero_centered, 0, 0, stream);
}

extern "C" int ix_gdn_scan_lens(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                                int io_dtype, long q_pitch, long k_pitch, long v_pitch, float* state_pool,
                                const int* cu_seqlens, const int* state_indices, long N, long H, long HV, long K, long V,
                                float scale, long tokens, long longest, const void* gate, long gate_stride_t,
                                const void* norm_weight, float norm_eps, int zero_centered, void* stream) {
  if (!o || tokens < 0 || longest < 0 || (gate && (!norm_weight || gate_stride_t < HV * V))) return IX_ERR_ARG;
  if (gate && !ix_gdn_norm_fits(o, io_dtype, K, V, gate, gate_stride_t, norm_weight)) return IX_DECLINED;
  return ix_gdn_scan_impl(q, k, v, g, beta, o, io_dtype, q_pitch, k_pitch, v_pitch, state_pool, cu_seqlens, state_indices, 0,
                          N, H, HV, K, V, scale, 0, (const bf16_t*)gate, gate_stride_t, (const bf16_t*)norm_weight, norm_eps,
                          zero_centered, tokens, longest, stream);
}

extern "C" int ix_gdn_layout(long N, long HV, long K, long V, int io_dtype, long chunk, long tokens, long longest) {
  if (N <= 0 || HV <= 0 || V <= 0 || K != 128) return 0;
  return ix_gdn_layout_for(N, HV, V, tokens, longest, io_dtype == IX_DT_BF16, chunk > 0);
}

// The stateless forward: every sequence starts from a zero state, which is not kept. chunk 0: the recurrence; chunk > 0:
// the boundary form, whose running state restarts every `chunk` tokens from the fp32 chain rounded to io_dtype.
extern "C" int ix_gdn_forward_lens(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                                   int io_dtype, long q_pitch, long k_pitch, long v_pitch, const int* cu_seqlens, long N,
                                   long H, long HV, long K, long V, float scale, long chunk, long tokens, long longest,
                                   const void* gate, long gate_stride_t, const void* norm_weight, float norm_eps,
                                   int zero_centered, void* stream) {
  if (!q || !k || !v || !g || !beta || !o || !cu_seqlens || tokens < 0 || longest < 0) return IX_ERR_ARG;
  if (N < 0 || H <= 0 || HV <= 0 || K <= 0 || V <= 0 || HV % H != 0 || chunk < 0) return IX_ERR_ARG;
  if (q_pitch < H * K || k_pitch < H * K || v_pitch < HV * V) return IX_ERR_ARG;
  if (gate && (!norm_weight || gate_stride_t < HV * V)) return IX_ERR_ARG;
  if (io_dtype != IX_DT_F32 && io_dtype != IX_DT_BF16) return IX_DECLINED;
  if (chunk % 16 || chunk > 0x7fffffffL) return IX_DECLINED;  // the restart falls on a tile's first token
  hipStream_t st = (hipStream_t)stream;
  const int layout = ix_gdn_layout(N, HV, K, V, io_dtype, chunk, tokens, longest);
  if (gate && (layout != IX_GDN_FOUR_TWO || !ix_gdn_norm_fits(o, io_dtype, K, V, gate, gate_stride_t, norm_weight)))
    return IX_DECLINED;  // the norm rides on two rows per lane only
  if (N == 0) return IX_OK;
  if (layout == IX_GDN_FOUR_TWO)
    return ix_gdn_quads(q, k, v, g, beta, o, io_dtype, q_pitch, k_pitch, v_pitch, nullptr, cu_seqlens, nullptr, N, (int)H,
                        (int)HV, (int)V, scale, 16, (const bf16_t*)gate, gate_stride_t, (const bf16_t*)norm_weight,
                        norm_eps, zero_centered, st);
  return ix_gdn_walk(q, k, v, g, beta, o, io_dtype, nullptr, cu_seqlens, nullptr, q_pitch, k_pitch, v_pitch, N, (int)H,
                     (int)HV, K, (int)V, scale, (int)chunk, layout == IX_GDN_FOUR_ONE ? 3 : 0, st);
}

extern "C" int ix_gdn_forward(const void* q, const void* k, const void* v, const float* g, const void* beta, void* o,
                              int io_dtype, long q_pitch, long k_pitch, long v_pitch, const int* cu_seqlens, long N, long H,
                              long HV, long K, long V, float scale, long chunk, const void* gate, long gate_stride_t,
                              const void* norm_weight, float norm_eps, int zero_centered, void* stream) {
  return ix_gdn_forward_lens(q, k, v, g, beta, o, io_dtype, q_pitch, k_pitch, v_pitch, cu_seqlens, N, H, HV, K, V, scale, chunk,
                             0, 0, gate, gate_stride_t, norm_weight, norm_eps, zero_centered, stream);
}

// ---------------------------------------------------------------------------------------------
// Preparation (gdn_ops.py:173-213 l2norm, :1197-1210 gating; fused form gdn_ops.py:513-558):
//   qn = io(x * (1 / sqrt(sum_k x_k^2 + 1e-6)))   sum: ix_tree8 over a lane's 8 squares, then the
//                                                 adjacent-pairwise tree over the K/8 lanes
//   g    = -exp(A_log[hv]) * softplus(a + dt_bias[hv])        fp32
//   beta = io(sigmoid(b))
template <int KS, typename TIO>
__global__ __launch_bounds__(256) void k_gdn_l2norm(const TIO* __restrict__ x, TIO* __restrict__ y, long rows,
                                                    int H, long x_pitch, float eps) {
  constexpr int K = KS * 8;
  constexpr int RPB = 256 / KS;
  const int sub = threadIdx.x % KS;
  const long row = (long)blockIdx.x * RPB + threadIdx.x / KS;
  const long rrow = row < rows ? row : rows - 1;
  float xv[8], sq[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    xv[i] = ix_ld(x + (rrow / H) * x_pitch + (rrow % H) * K + sub * 8 + i);
    sq[i] = xv[i] * xv[i];
  }
  const float s = ix_lane_tree<KS>(ix_tree8(sq));
  const float rn = ix_rsqrt_ieee(s + eps);
  if (row >= rows) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) ix_st(y + row * K + sub * 8 + i, xv[i] * rn);
}

template <typename TIO>
__global__ __launch_bounds__(256) void k_gdn_gate(const TIO* __restrict__ a, long a_pitch,
                                                  const TIO* __restrict__ b, long b_pitch,
                                                  const float* __restrict__ A_log,
                                                  const float* __restrict__ dt_bias, float* __restrict__ g,
                                                  TIO* __restrict__ beta, long n, int HV, int exp_bf16) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const long t = i / HV;
  const int hv = (int)(i - t * HV);
  const float sp = ix_softplus(ix_ld(a + t * a_pitch + hv) + dt_bias[hv]);
  float ea = ix_exp(A_log[hv]);
  if (exp_bf16) ea = ix_bf2f(ix_f2bf(ea));  // a bf16 parameter's exp() is a bf16 value (the eager form's rounding)
  const float neg_ea = -ea;
  g[i] = neg_ea * sp;
  ix_st(beta + i, ix_sigmoid(ix_ld(b + t * b_pitch + hv)));
}

extern "C" int ix_gdn_l2norm(const void* x, long x_pitch, void* y, int io_dtype, long tokens, long H, long K,
                             float eps, void* stream) {
  if (!x || !y || tokens < 0 || H <= 0 || K <= 0 || x_pitch < H * K) return IX_ERR_ARG;
  const long rows = tokens * H;
  if (io_dtype != IX_DT_F32 && io_dtype != IX_DT_BF16) return IX_DECLINED;
  if (rows == 0) return IX_OK;
  hipStream_t st = (hipStream_t)stream;
#define IX_L2_CASE(KSV)                                                                                          \
  if (K == KSV * 8) {                                                                                            \
    const long grid = (rows + (256 / KSV) - 1) / (256 / KSV);                                                    \
    if (grid > 0x7fffffffL) return IX_DECLINED;                                                                  \
    if (io_dtype == IX_DT_BF16)                                                                                  \
      hipLaunchKernelGGL((k_gdn_l2norm<KSV, bf16_t>), dim3((unsigned)grid), dim3(256), 0, st, (const bf16_t*)x, \
                         (bf16_t*)y, rows, (int)H, x_pitch, eps);                                                \
    else                                                                                                         \
      hipLaunchKernelGGL((k_gdn_l2norm<KSV, float>), dim3((unsigned)grid), dim3(256), 0, st, (const float*)x,   \
                         (float*)y, rows, (int)H, x_pitch, eps);                                                 \
    return ix_launch_status();                                                                                   \
  }
  IX_L2_CASE(4)
  IX_L2_CASE(8)
  IX_L2_CASE(16)
  IX_L2_CASE(32)
#undef IX_L2_CASE
  return IX_DECLINED;
}

extern "C" int ix_gdn_gate(const void* a, long a_pitch, const void* b, long b_pitch, const float* A_log,
                           const float* dt_bias, float* g, void* beta, int io_dtype, long tokens, long HV,
                           int exp_dtype, void* stream) {
  if (!a || !b || !A_log || !dt_bias || !g || !beta || tokens < 0 || HV <= 0 || a_pitch < HV || b_pitch < HV)
    return IX_ERR_ARG;
  if (io_dtype != IX_DT_F32 && io_dtype != IX_DT_BF16) return IX_DECLINED;
  if (exp_dtype != IX_DT_F32 && exp_dtype != IX_DT_BF16) return IX_DECLINED;
  const int exp_bf16 = exp_dtype == IX_DT_BF16;
  const long n = tokens * HV;
  if (n == 0) return IX_OK;
  const long grid = (n + 255) / 256;
  if (grid > 0x7fffffffL) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  if (io_dtype == IX_DT_BF16)
    hipLaunchKernelGGL((k_gdn_gate<bf16_t>), dim3((unsigned)grid), dim3(256), 0, st, (const bf16_t*)a, a_pitch,
                       (const bf16_t*)b, b_pitch, A_log, dt_bias, g, (bf16_t*)beta, n, (int)HV, exp_bf16);
  else
    hipLaunchKernelGGL((k_gdn_gate<float>), dim3((unsigned)grid), dim3(256), 0, st, (const float*)a, a_pitch,
                       (const float*)b, b_pitch, A_log, dt_bias, g, (float*)beta, n, (int)HV, exp_bf16);
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// Open-chunk bookkeeping of the boundary (cpr) engine state (gdn_cpr_scatter.py:24-76; eager form
// gdn_cpr_state.py decode): lane n appends this step's prepared k, v, g, beta to the open-chunk buffers of its
// pool row at column pos[row] % C, then pos[row] += 1 (not for row 0, which absorbs padded lanes), and marks the
// row due for a boundary pass when its position has reached a multiple of C. One workgroup per lane; a live row
// appears at most once per step.
template <typename TIO>
__global__ __launch_bounds__(256) void k_gdn_cpr_scatter(const TIO* __restrict__ k, long k_pitch,
                                                         const TIO* __restrict__ v, long v_pitch,
                                                         const float* __restrict__ g, const TIO* __restrict__ beta,
                                                         const int* __restrict__ rows, int64_t* __restrict__ pos,
                                                         TIO* __restrict__ k_buf, TIO* __restrict__ v_buf,
                                                         float* __restrict__ g_buf, TIO* __restrict__ b_buf,
                                                         int* __restrict__ due, int HK, int HVV, int HV, int C) {
  const int n = blockIdx.x;
  const int row = rows[n];
  const int64_t p = pos[row];
  const int col = (int)(p % C);
  __syncthreads();  // every lane has read the position before lane 0 advances it
  const long slot = (long)row * C + col;
  for (int i = threadIdx.x; i < HK; i += 256) k_buf[slot * HK + i] = k[(long)n * k_pitch + i];
  for (int i = threadIdx.x; i < HVV; i += 256) v_buf[slot * HVV + i] = v[(long)n * v_pitch + i];
  for (int i = threadIdx.x; i < HV; i += 256) {
    g_buf[slot * HV + i] = g[(long)n * HV + i];
    b_buf[slot * HV + i] = beta[(long)n * HV + i];
  }
  if (threadIdx.x == 0 && row > 0) {
    pos[row] = p + 1;
    due[row] = ((p + 1) % C == 0) ? row : 0;
  }
}

extern "C" int ix_gdn_cpr_scatter(const void* k, long k_pitch, const void* v, long v_pitch, const float* g,
                                  const void* beta, const int* rows, int64_t* pos, void* k_buf, void* v_buf,
                                  float* g_buf, void* b_buf, int* due, int io_dtype, long N, long H, long K, long HV,
                                  long V, long C, void* stream) {
  if (!k || !v || !g || !beta || !rows || !pos || !k_buf || !v_buf || !g_buf || !b_buf || !due) return IX_ERR_ARG;
  if (N < 0 || H <= 0 || K <= 0 || HV <= 0 || V <= 0 || C <= 0 || k_pitch < H * K || v_pitch < HV * V)
    return IX_ERR_ARG;
  if (io_dtype != IX_DT_F32 && io_dtype != IX_DT_BF16) return IX_DECLINED;
  if (N == 0) return IX_OK;
  if (N > 0x7fffffffL) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  if (io_dtype == IX_DT_BF16)
    hipLaunchKernelGGL(k_gdn_cpr_scatter<bf16_t>, dim3((unsigned)N), dim3(256), 0, st, (const bf16_t*)k, k_pitch,
                       (const bf16_t*)v, v_pitch, g, (const bf16_t*)beta, rows, pos, (bf16_t*)k_buf, (bf16_t*)v_buf,
                       g_buf, (bf16_t*)b_buf, due, (int)(H * K), (int)(HV * V), (int)HV, (int)C);
  else
    hipLaunchKernelGGL(k_gdn_cpr_scatter<float>, dim3((unsigned)N), dim3(256), 0, st, (const float*)k, k_pitch,
                       (const float*)v, v_pitch, g, (const float*)beta, rows, pos, (float*)k_buf, (float*)v_buf, g_buf,
                       (float*)b_buf, due, (int)(H * K), (int)(HV * V), (int)HV, (int)C);
  return ix_launch_status();
}

// The hand-off after a boundary pass (gdn_cpr_state.py:602-646): for every pool row marked due, the running state
// becomes the snapshot of the fp32 chain (rounded to the wire dtype and widened back), and the mark is cleared.
__global__ __launch_bounds__(256) void k_gdn_cpr_handoff(const float* __restrict__ entry, float* __restrict__ running,
                                                         int* __restrict__ due, long elems, int snap_bf16) {
  const int row = blockIdx.y;
  if (due[row] <= 0) return;
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i < elems) {
    float4 x = *reinterpret_cast<const float4*>(entry + (long)row * elems + i);
    if (snap_bf16) { x.x = ix_rbf(x.x); x.y = ix_rbf(x.y); x.z = ix_rbf(x.z); x.w = ix_rbf(x.w); }
    *reinterpret_cast<float4*>(running + (long)row * elems + i) = x;
  }
}
__global__ __launch_bounds__(256) void k_gdn_cpr_clear_due(int* __restrict__ due, int rows) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < rows) due[i] = 0;
}

extern "C" int ix_gdn_cpr_handoff(const float* entry_state, float* running_state, int* due, long rows, long elems,
                                  int snapshot_dtype, void* stream) {
  if (!entry_state || !running_state || !due || rows < 0 || elems <= 0) return IX_ERR_ARG;
  if (snapshot_dtype != IX_DT_F32 && snapshot_dtype != IX_DT_BF16) return IX_DECLINED;
  if ((elems % 4) || !ix_aligned(entry_state, 16) || !ix_aligned(running_state, 16)) return IX_DECLINED;
  if (rows == 0) return IX_OK;
  const long gx = (elems / 4 + 255) / 256;
  if (rows > 65535 || gx > 0x7fffffffL) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_gdn_cpr_handoff, dim3((unsigned)gx, (unsigned)rows), dim3(256), 0, st, entry_state,
                     running_state, due, elems, snapshot_dtype == IX_DT_BF16);
  // the marks are cleared by a second launch: every workgroup of the first reads its row's mark
  hipLaunchKernelGGL(k_gdn_cpr_clear_due, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, st, due, (int)rows);
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// Slot ids -> state-pool rows for a decode batch in one launch (gdn_cpr_rows.py:29-46, the fused form of
// gdn_recurrent_state.py:271-284): with a map, row = slot2row[clamp(slot, 0, map_n - 1)]; without one (the
// engine's block ids are the rows), row = slot if 0 <= slot < blocks else 0. Optionally the same launch stamps the
// rows' last-use clock (gdn_recurrent_state.py decode: clock += 1; last_used[rows] = clock). One workgroup, so
// every lane reads the clock before lane 0 advances it.
template <typename TS>
__global__ __launch_bounds__(256) void k_gdn_resolve_rows(const TS* __restrict__ slots, long n,
                                                          const int64_t* __restrict__ slot2row, long map_n,
                                                          long blocks, int64_t* __restrict__ rows64,
                                                          int* __restrict__ rows32, int64_t* __restrict__ last_used,
                                                          int64_t* __restrict__ clock) {
  const int64_t stamp = clock ? clock[0] + 1 : 0;
  for (long i = threadIdx.x; i < n; i += 256) {
    int64_t sl = (int64_t)slots[i];
    int64_t r;
    if (slot2row) {
      sl = sl < 0 ? 0 : (sl > map_n - 1 ? map_n - 1 : sl);
      r = slot2row[sl];
    } else {
      r = (sl >= 0 && sl < blocks) ? sl : 0;
    }
    if (rows64) rows64[i] = r;
    rows32[i] = (int)r;
    if (last_used) last_used[r] = stamp;
  }
  __syncthreads();
  if (clock && threadIdx.x == 0) clock[0] = stamp;
}

extern "C" int ix_gdn_resolve_rows(const void* slots, int slots_i64, long n, const int64_t* slot2row, long map_n,
                                   long blocks, int64_t* rows64, int* rows32, int64_t* last_used, int64_t* clock,
                                   void* stream) {
  if (n < 0 || (n > 0 && (!slots || !rows32))) return IX_ERR_ARG;
  if (slot2row ? map_n <= 0 : blocks <= 0) return IX_ERR_ARG;
  if ((last_used == nullptr) != (clock == nullptr)) return IX_ERR_ARG;
  if (n == 0 && !clock) return IX_OK;
  hipStream_t st = (hipStream_t)stream;
  if (slots_i64)
    hipLaunchKernelGGL(k_gdn_resolve_rows<int64_t>, dim3(1), dim3(256), 0, st, (const int64_t*)slots, n, slot2row,
                       map_n, blocks, rows64, rows32, last_used, clock);
  else
    hipLaunchKernelGGL(k_gdn_resolve_rows<int>, dim3(1), dim3(256), 0, st, (const int*)slots, n, slot2row, map_n,
                       blocks, rows64, rows32, last_used, clock);
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// What a prefill does to a layer's tables and pools in front of its kernels (gdn_recurrent_state.py prefill: slot-map scatter,
// use stamps, fresh rows zeroed), in one launch and from one upload: ten launches and copies of 4 to 5 us each before, none
// of which has work to speak of (8192 tokens through one layer 1088 -> 1047 us, the l2norm folded into the convolution with it).
// Workgroup 0 edits the tables (it alone reads the clock before it advances it), the others zero IX_GDN_ZERO floats each of a
// fresh row in the pools. The null row is zeroed once, however many sequences start no row.
#define IX_GDN_ZERO 8192
__global__ __launch_bounds__(256) void k_gdn_prefill_begin(const int64_t* __restrict__ map_edits, int edits,
                                                           const int64_t* __restrict__ stamps, int stamped, long advance,
                                                           const int* __restrict__ fresh, int N, int64_t* __restrict__ slot2row,
                                                           long map_n, int64_t* __restrict__ last_used,
                                                           int64_t* __restrict__ clock, float* __restrict__ pool,
                                                           float* __restrict__ pool2, int64_t* __restrict__ pos, long pool_rows,
                                                           long row_floats, int per_row) {
  const int tid = threadIdx.x;
  if (blockIdx.x == 0) {
    for (int i = tid; i < edits; i += 256) {
      const int64_t slot = map_edits[i], row = map_edits[edits + i];
      if (slot >= 0 && slot < map_n) slot2row[slot] = row;
    }
    const int64_t now = clock ? clock[0] : 0;
    for (int i = tid; i < stamped; i += 256) {
      const int64_t row = stamps[i];
      if (row >= 0 && row < pool_rows) last_used[row] = now + stamps[stamped + i];
    }
    if (pos) {
      for (int i = tid; i < N; i += 256)
        if (fresh[i] >= 0 && fresh[i] < pool_rows) pos[fresh[i]] = 0;
      if (tid == 0) pos[0] = 0;  // the null row's
    }
    __syncthreads();
    if (clock && tid == 0) clock[0] = now + advance;
    return;
  }
  const long at = blockIdx.x - 1;
  const int n = (int)(at / per_row);
  const int row = fresh[n];
  if (row < 0 || row >= pool_rows) return;
  if (row == 0)
    for (int j = 0; j < n; ++j)
      if (fresh[j] == 0) return;
  const long lo = at % per_row * (long)IX_GDN_ZERO, hi = min(row_floats, lo + IX_GDN_ZERO);
  for (long i = lo + 4 * tid; i < hi; i += 1024) {  // row_floats % 4 == 0
    *reinterpret_cast<float4*>(pool + row * row_floats + i) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (pool2) *reinterpret_cast<float4*>(pool2 + row * row_floats + i) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
}

extern "C" int ix_gdn_prefill_begin(const int64_t* map_edits, long edits, const int64_t* stamps, long stamped, long advance,
                                    const int* fresh, long N, int64_t* slot2row, long map_n, int64_t* last_used,
                                    int64_t* clock, float* pool, float* pool2, int64_t* pos, long pool_rows, long row_floats,
                                    void* stream) {
  if (edits < 0 || stamped < 0 || N < 0 || advance < 0 || pool_rows <= 0 || row_floats <= 0 || !pool) return IX_ERR_ARG;
  if ((edits > 0 && (!map_edits || !slot2row || map_n <= 0)) || (stamped > 0 && (!stamps || !last_used || !clock)) ||
      (N > 0 && !fresh))
    return IX_ERR_ARG;
  if (row_floats % 4 || !ix_aligned(pool, 16) || (pool2 && !ix_aligned(pool2, 16))) return IX_DECLINED;
  const long per_row = (row_floats + IX_GDN_ZERO - 1) / IX_GDN_ZERO;
  if (edits > 0x7fffffffL || stamped > 0x7fffffffL || N * per_row >= 0x7fffffffL) return IX_DECLINED;
  hipLaunchKernelGGL(k_gdn_prefill_begin, dim3((unsigned)(1 + N * per_row)), dim3(256), 0, (hipStream_t)stream, map_edits,
                     (int)edits, stamps, (int)stamped, advance, fresh, (int)N, slot2row, map_n, last_used, clock, pool, pool2,
                     pos, pool_rows, row_floats, (int)per_row);
  return ix_launch_status();
}

// ---------------------------------------------------------------------------------------------
// Causal depthwise conv of width W <= 8 over packed tokens (gdn_ops.py:74-170):
//   acc = 0; for i = 0..W-1: acc = acc + w[d,i] * xp[t+i]   (multiply rounded, add rounded)
//   acc = acc + bias[d]; acc = acc * sigmoid(acc); y = bf16(acc)
// xp = [W-1 previous inputs (oldest first), from the state pool row or zeros] ++ x. A decode
// step is the same kernel with one token per sequence. The final state (the last W-1 inputs)
// is written by a second kernel so an in-place pool row is never read and written in one launch.
__device__ __forceinline__ int ix_seq_of(const int* __restrict__ cu, int N, int t) {
  int lo = 0, hi = N;  // largest n with cu[n] <= t
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu[mid] <= t) lo = mid; else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ float ix_conv_xp(const bf16_t* __restrict__ x, long x_pitch,
                                            const bf16_t* __restrict__ pool, int srow, int t_begin, int rel, long D,
                                            int d, int W) {
  // rel: position relative to the sequence start; negative -> history slot W-1+rel
  if (rel >= 0) return ix_bf2f(x[(long)(t_begin + rel) * x_pitch + d]);
  if (srow <= 0) return 0.0f;
  return ix_bf2f(pool[((long)srow * D + d) * (W - 1) + (W - 1 + rel)]);
}

__global__ __launch_bounds__(256) void k_gdn_conv(const bf16_t* __restrict__ x, long x_pitch,
                                                  const bf16_t* __restrict__ w,
                                                  const bf16_t* __restrict__ bias, bf16_t* __restrict__ y,
                                                  const bf16_t* __restrict__ pool, const int* __restrict__ cu,
                                                  const int* __restrict__ rows_in, int N, long D, int W,
                                                  int silu, long total) {
  // Two grid dimensions: one dimension may not exceed 2^32 threads, and a packed prefill does.
  const long i = ((long)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int t = (int)(i / D);
  const int d = (int)(i % D);
  const int n = ix_seq_of(cu, N, t);
  const int t_begin = cu[n];
  const int rel = t - t_begin;
  const int srow = rows_in ? rows_in[n] : 0;
  float acc = 0.0f;
  for (int j = 0; j < W; ++j) {
    const float xv = ix_conv_xp(x, x_pitch, pool, srow, t_begin, rel - (W - 1) + j, D, d, W);
    const float p = ix_bf2f(w[(long)d * W + j]) * xv;
    acc = acc + p;
  }
  if (bias) acc = acc + ix_bf2f(bias[d]);
  if (silu) acc = acc * ix_sigmoid(acc);
  y[i] = ix_f2bf(acc);
}

// Eight consecutive channels of four consecutive tokens per thread: 16-byte loads and stores, and inside a
// sequence each input row is loaded once for the four windows that cover it. Per channel the arithmetic is that
// of k_gdn_conv, statement for statement, so the two kernels agree bit for bit (a NaN keeps its payload here).
template <int W>
__device__ __forceinline__ void ix_conv8_finish(const float (&xv)[W][8], const float (&wv)[8][W], bool has_bias,
                                                const float (&bv)[8], int silu, bf16_t* __restrict__ yrow) {
  uint32_t out[4];
#pragma unroll
  for (int c = 0; c < 8; c += 2) {
    float r2[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      float acc = 0.0f;
#pragma unroll
      for (int j = 0; j < W; ++j) {
        const float p = wv[c + e][j] * xv[j][c + e];
        acc = acc + p;
      }
      if (has_bias) acc = acc + bv[c + e];
      if (silu) acc = acc * ix_sigmoid(acc);
      r2[e] = acc;
    }
    out[c >> 1] = ix_pack_bf2_hw(r2[0], r2[1]);
  }
  *reinterpret_cast<uint4*>(yrow) = make_uint4(out[0], out[1], out[2], out[3]);
}


// The l2norm of a q or k head (K = 128: sixteen lanes of eight channels) on the bf16 values the convolution just
// rounded -- k_gdn_l2norm<16>'s expression on what it would have read back: squares, ix_tree8, the adjacent-pairwise
// tree over the sixteen lanes, one IEEE rsqrt, bf16(x * r). Every lane of the sixteen must be here.
__device__ __forceinline__ void ix_l2norm8_of16(bf16_t* __restrict__ yrow, float eps) {
  float v8[8], sq[8];
  ix_unpack8(*reinterpret_cast<const uint4*>(yrow), v8);
#pragma unroll
  for (int i = 0; i < 8; ++i) sq[i] = v8[i] * v8[i];
  const float ssum = ix_lane_tree<16>(ix_tree8(sq));
  const float rn = ix_rsqrt_ieee(ssum + eps);
  if (ssum < __builtin_inff()) {
    // every value is finite and so is every product: the hardware pack-convert rounds them as ix_f2bf does
    *reinterpret_cast<uint4*>(yrow) =
        make_uint4(ix_pack_bf2_hw(v8[0] * rn, v8[1] * rn), ix_pack_bf2_hw(v8[2] * rn, v8[3] * rn),
                   ix_pack_bf2_hw(v8[4] * rn, v8[5] * rn), ix_pack_bf2_hw(v8[6] * rn, v8[7] * rn));
    return;
  }
  // an infinity or a NaN among the head's values: products can be NaN, which ix_f2bf canonicalises
  __attribute__((aligned(16))) bf16_t out[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) out[i] = ix_f2bf(v8[i] * rn);
  *reinterpret_cast<uint4*>(yrow) = *reinterpret_cast<const uint4*>(out);
}

// NORM: channels below qk_channels are q and k heads of 128 and leave normalised (ix_gdn_conv_l2norm); a head's sixteen
// threads are consecutive and share the token group, so they take the same path through the kernel.
template <int W, int TOK, bool NORM>
__global__ __launch_bounds__(256) void k_gdn_conv8(const bf16_t* __restrict__ x, long x_pitch,
                                                   const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias,
                                                   bf16_t* __restrict__ y, const bf16_t* __restrict__ pool,
                                                   const int* __restrict__ cu, const int* __restrict__ rows_in,
                                                   int N, long D, int silu, int T, long total, long qk_channels,
                                                   float eps, unsigned run_blocks, unsigned run_groups) {
  const long D8 = D >> 3;
  long i;
  if (run_blocks) {
    // Consecutive token groups of one 2048-channel block on one XCD, one after the other: the W - 1 rows a group
    // shares with the group before it are then still in that XCD's L2 (dealt round-robin, neighbouring groups sit
    // on different XCDs and every shared row is fetched twice). The host chose this only for D8 % 256 == 0.
    unsigned pos;
    if (!ix_xcd_run_position(blockIdx.x, run_blocks, &pos)) return;
    i = (long)(pos % run_groups) * D8 + (long)(pos / run_groups) * 256 + threadIdx.x;
  } else {
    i = ((long)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
  }
  if (i >= total) return;
  const int t0 = (int)(i / D8) * TOK;
  const int d = (int)(i % D8) * 8;
  float wv[8][W], bv[8];
  {
    // 8 channels x W taps are 8 W consecutive elements (the host checked the alignment): W 16-byte loads
    static_assert(W == 4, "the unpacking below assumes four taps");
    const uint4* wp = reinterpret_cast<const uint4*>(w + (long)d * W);
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2) {
      float t8[8];
      ix_unpack8(wp[c2], t8);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        wv[2 * c2][j] = t8[j];
        wv[2 * c2 + 1][j] = t8[4 + j];
      }
    }
    // the channels' biases once per thread, not once per output
    if (bias) {
      ix_unpack8(*reinterpret_cast<const uint4*>(bias + d), bv);
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) bv[c] = 0.0f;
    }
  }
  const bool has_bias = bias != nullptr;
  const int n0 = ix_seq_of(cu, N, t0);
  const int b0 = cu[n0], e0 = cu[n0 + 1];
  if (t0 - (W - 1) >= b0 && t0 + TOK <= e0) {
    // all TOK windows lie inside one sequence: TOK + W - 1 rows serve TOK outputs
    // the rows stay packed (4 registers each) until a window needs them
    uint4 xr[TOK + W - 1];
#pragma unroll
    for (int r = 0; r < TOK + W - 1; ++r)
      xr[r] = *reinterpret_cast<const uint4*>(x + (long)(t0 - (W - 1) + r) * x_pitch + d);
#pragma unroll
    for (int q = 0; q < TOK; ++q) {
      float xv[W][8];
#pragma unroll
      for (int j = 0; j < W; ++j) ix_unpack8(xr[q + j], xv[j]);
      if constexpr (NORM) {
        __attribute__((aligned(16))) bf16_t yv[8];
        ix_conv8_finish<W>(xv, wv, has_bias, bv, silu, yv);
        if (d < qk_channels) ix_l2norm8_of16(yv, eps);
        *reinterpret_cast<uint4*>(y + (long)(t0 + q) * D + d) = *reinterpret_cast<const uint4*>(yv);
      } else {
        ix_conv8_finish<W>(xv, wv, has_bias, bv, silu, y + (long)(t0 + q) * D + d);
      }
    }
    return;
  }
  for (int q = 0; q < TOK; ++q) {
    const int t = t0 + q;
    if (t >= T) break;
    const int n = ix_seq_of(cu, N, t);
    const int t_begin = cu[n];
    const int rel = t - t_begin;
    const int srow = rows_in ? rows_in[n] : 0;
    float xv[W][8];
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const int r = rel - (W - 1) + j;
      if (r >= 0) {
        ix_unpack8(*reinterpret_cast<const uint4*>(x + (long)(t_begin + r) * x_pitch + d), xv[j]);
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          xv[j][c] = srow > 0 ? ix_bf2f(pool[((long)srow * D + d + c) * (W - 1) + (W - 1 + r)]) : 0.0f;
      }
    }
    if constexpr (NORM) {
      __attribute__((aligned(16))) bf16_t yv[8];
      ix_conv8_finish<W>(xv, wv, has_bias, bv, silu, yv);
      if (d < qk_channels) ix_l2norm8_of16(yv, eps);
      *reinterpret_cast<uint4*>(y + (long)t * D + d) = *reinterpret_cast<const uint4*>(yv);
    } else {
      ix_conv8_finish<W>(xv, wv, has_bias, bv, silu, y + (long)t * D + d);
    }
  }
}

__global__ __launch_bounds__(256) void k_gdn_conv_state(const bf16_t* __restrict__ x, long x_pitch,
                                                        bf16_t* __restrict__ pool,
                                                        const int* __restrict__ cu,
                                                        const int* __restrict__ rows_in,
                                                        const int* __restrict__ rows_out, int N, long D, int W) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)N * D) return;
  const int n = (int)(i / D);
  const int d = (int)(i % D);
  const int orow = rows_out[n];
  if (orow <= 0) return;
  const int t_begin = cu[n], len = cu[n + 1] - t_begin;
  const int srow = rows_in ? rows_in[n] : 0;
  bf16_t tmp[8];
  for (int j = 0; j < W - 1; ++j) {
    // new history slot j holds the input at relative position len - (W-1) + j
    const float xv = ix_conv_xp(x, x_pitch, pool, srow, t_begin, len - (W - 1) + j, D, d, W);
    tmp[j] = ix_f2bf(xv);  // exact: the value is a bf16 already
  }
  for (int j = 0; j < W - 1; ++j) pool[((long)orow * D + d) * (W - 1) + j] = tmp[j];
}

static int ix_gdn_conv_impl(const void* x, long x_pitch, const void* weight, const void* bias, void* y,
                            void* conv_pool, const int* cu_seqlens, const int* state_rows_in,
                            const int* state_rows_out, long N, long total_tokens, long D, long W, int silu,
                            long qk_channels, float eps, void* stream) {
  if (!x || !weight || !y || !cu_seqlens || N < 0 || total_tokens < 0 || D <= 0 || x_pitch < D) return IX_ERR_ARG;
  if (W < 1 || W > 8) return IX_DECLINED;
  if ((state_rows_in || state_rows_out) && !conv_pool) return IX_ERR_ARG;
  if (total_tokens > 0x7fffffffL || N > 0x7fffffffL) return IX_DECLINED;
  hipStream_t st = (hipStream_t)stream;
  const long total = total_tokens * D;
  if (total > 0 && N > 0) {
    const bool vec8 = (W == 4) && (D % 8 == 0) && (x_pitch % 8 == 0) && ix_aligned(x, 16) && ix_aligned(y, 16) &&
                      ix_aligned(weight, 16) && (!bias || ix_aligned(bias, 16));
    // Outputs per thread: long sequences amortise the W - 1 rows of history over 16 outputs; short ones (a decode
    // step has one token per sequence) keep one output per thread so the launch stays wide. Every output is
    // computed by the same expression whichever is chosen.
    if (qk_channels > 0 && !vec8) return IX_DECLINED;  // the normalising form is the eight-channel kernel's
    const long avg_len = total_tokens / N;
    // The normalising form stops at 8: with 16 its registers leave two waves per SIMD and the launch takes a quarter
    // longer than the plain one; with 8 it takes the same time (1.17 ms for 163,840 tokens of 8192 channels).
    const int TOK = !vec8 ? 1 : avg_len >= 64 ? (qk_channels > 0 ? 8 : 16) : avg_len >= 8 ? 4 : 1;
    const long work = vec8 ? ((total_tokens + TOK - 1) / TOK) * (D / 8) : total;
    const long blocks = (work + 255) / 256;
    // the XCD-run order for long sequences whose channel count fills whole workgroups
    const bool runs = vec8 && TOK > 1 && (D / 8) % 256 == 0 && blocks < (1L << 30);
    const unsigned run_blocks = runs ? (unsigned)blocks : 0u;
    const unsigned run_groups = runs ? (unsigned)((total_tokens + TOK - 1) / TOK) : 1u;
    const long gx = runs ? (long)ix_xcd_run_grid(run_blocks) : blocks < (1L << 22) ? blocks : (1L << 22);
    const long gy = runs ? 1 : (blocks + gx - 1) / gx;
    if (gy > 65535) return IX_DECLINED;
#define IX_CONV8(TOK_, NORM_)                                                                                       \
  hipLaunchKernelGGL((k_gdn_conv8<4, TOK_, NORM_>), dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, st,             \
                     (const bf16_t*)x, x_pitch, (const bf16_t*)weight, (const bf16_t*)bias, (bf16_t*)y,             \
                     (const bf16_t*)conv_pool, cu_seqlens, state_rows_in, (int)N, D, silu, (int)total_tokens, work, \
                     qk_channels, eps, run_blocks, run_groups)
    if (vec8 && qk_channels > 0) {
      if (TOK == 8) IX_CONV8(8, true);
      else if (TOK == 4) IX_CONV8(4, true);
      else IX_CONV8(1, true);
    } else if (vec8) {
      if (TOK == 16) IX_CONV8(16, false);
      else if (TOK == 4) IX_CONV8(4, false);
      else IX_CONV8(1, false);
    }
#undef IX_CONV8
    else
      hipLaunchKernelGGL(k_gdn_conv, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, st, (const bf16_t*)x, x_pitch,
                         (const bf16_t*)weight, (const bf16_t*)bias, (bf16_t*)y, (const bf16_t*)conv_pool, cu_seqlens,
                         state_rows_in, (int)N, D, (int)W, silu, total);
  }
  if (state_rows_out && N > 0 && W > 1) {
    const long grid = (N * D + 255) / 256;
    if (grid > 0x7fffffffL) return IX_DECLINED;
    hipLaunchKernelGGL(k_gdn_conv_state, dim3((unsigned)grid), dim3(256), 0, st, (const bf16_t*)x, x_pitch,
                       (bf16_t*)conv_pool, cu_seqlens, state_rows_in, state_rows_out, (int)N, D, (int)W);
  }
  return ix_launch_status();
}

extern "C" int ix_gdn_conv(const void* x, long x_pitch, const void* weight, const void* bias, void* y,
                           void* conv_pool, const int* cu_seqlens, const int* state_rows_in,
                           const int* state_rows_out, long N, long total_tokens, long D, long W, int silu,
                           void* stream) {
  return ix_gdn_conv_impl(x, x_pitch, weight, bias, y, conv_pool, cu_seqlens, state_rows_in, state_rows_out, N,
                          total_tokens, D, W, silu, 0, 0.0f, stream);
}

// ix_gdn_conv with the l2norm of the q and k heads folded into its epilogue: channels [0, qk_channels) of y are heads of
// K = 128 and leave normalised (the bits of ix_gdn_conv followed by ix_gdn_l2norm over those columns), the rest (v) as
// ix_gdn_conv leaves them. Serves the eight-channel form only: W = 4, D and x_pitch multiples of 8, 16-byte aligned
// operands, qk_channels a multiple of 128; bf16.
extern "C" int ix_gdn_conv_l2norm(const void* x, long x_pitch, const void* weight, const void* bias, void* y,
                                  void* conv_pool, const int* cu_seqlens, const int* state_rows_in,
                                  const int* state_rows_out, long N, long total_tokens, long D, long W, int silu,
                                  long qk_channels, long K, float eps, void* stream) {
  if (qk_channels <= 0 || qk_channels > D || K <= 0) return IX_ERR_ARG;
  if (K != 128 || (qk_channels % 128) || (D % 128) || W != 4) return IX_DECLINED;
  return ix_gdn_conv_impl(x, x_pitch, weight, bias, y, conv_pool, cu_seqlens, state_rows_in, state_rows_out, N,
                          total_tokens, D, W, silu, qk_channels, eps, stream);
}

// ---------------------------------------------------------------------------------------------
// Everything a decode step does in front of the scan, in ONE launch (one token per sequence): the width-4 conv on the
// row's stored window with the window slid in place, the l2norm of the q and k heads, the gating. It replaces four
// launches (k_gdn_conv8<4, 1>, k_gdn_conv_state, k_gdn_l2norm<16>, k_gdn_gate: 4 - 8 us each at batch 64, all of it
// launch latency) and computes every value by the same statements:
//   conv    ix_conv8_finish on [h0, h1, h2, x] -> eight packed bf16 (k_gdn_conv8's expression)
//   window  [h1, h2, x] back to the same pool row (k_gdn_conv_state's values; a thread owns its eight channels' window,
//           reads it before it writes it, and nobody else touches it: no second launch is needed when the row a
//           sequence reads is the row it writes)
//   l2norm  on the bf16 values the conv stored, ix_tree8 + ix_lane_tree<16> (k_gdn_l2norm<16>'s expression): a head of
//           128 channels is 16 consecutive threads
//   gate    k_gdn_gate's two expressions, by the first HV threads of the sequence's first workgroup
// Layout: thread = eight consecutive channels of one sequence; workgroup = 2048 channels; grid = (D / 2048, N).
// y [N, D] receives normalised q and k (channels < 2 H K) and the conv's v behind them. A row <= 0 (a padded lane)
// reads a zero window and writes none.
__global__ __launch_bounds__(256) void k_gdn_decode_prep(const bf16_t* __restrict__ x, long x_pitch,
                                                         const bf16_t* __restrict__ a, long a_pitch,
                                                         const bf16_t* __restrict__ b, long b_pitch,
                                                         const bf16_t* __restrict__ w, const bf16_t* __restrict__ bias,
                                                         const float* __restrict__ A_log,
                                                         const float* __restrict__ dt_bias, bf16_t* __restrict__ pool,
                                                         const int* __restrict__ rows, bf16_t* __restrict__ y,
                                                         float* __restrict__ g, bf16_t* __restrict__ beta, long D,
                                                         int qk_channels, int HV, int silu, float eps) {
  constexpr int W = 4;
  const int n = blockIdx.y;
  const int d = (blockIdx.x * 256 + threadIdx.x) * 8;
  const int row = rows[n];
  if (blockIdx.x == 0) {
    for (int hv = threadIdx.x; hv < HV; hv += 256) {
      const float sp = ix_softplus(ix_ld(a + (long)n * a_pitch + hv) + dt_bias[hv]);
      const float neg_ea = -ix_exp(A_log[hv]);
      g[(long)n * HV + hv] = neg_ea * sp;
      ix_st(beta + (long)n * HV + hv, ix_sigmoid(ix_ld(b + (long)n * b_pitch + hv)));
    }
  }
  // whole 16-lane groups leave together (D is a multiple of 128): the lane tree below stays inside live groups
  if (d >= D) return;
  float wv[8][W], bv[8];
  {
    const uint4* wp = reinterpret_cast<const uint4*>(w + (long)d * W);
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2) {
      float t8[8];
      ix_unpack8(wp[c2], t8);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        wv[2 * c2][j] = t8[j];
        wv[2 * c2 + 1][j] = t8[4 + j];
      }
    }
    if (bias) {
      ix_unpack8(*reinterpret_cast<const uint4*>(bias + d), bv);
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) bv[c] = 0.0f;
    }
  }
  // the window of the thread's eight channels: 8 x 3 consecutive bf16 of the pool row
  bf16_t hist[8 * (W - 1)];
  bf16_t* hp = pool + ((long)(row > 0 ? row : 0) * D + d) * (W - 1);
  if (row > 0) {
    const uint4* h4 = reinterpret_cast<const uint4*>(hp);
#pragma unroll
    for (int i = 0; i < 3; ++i) reinterpret_cast<uint4*>(hist)[i] = h4[i];
  } else {
#pragma unroll
    for (int i = 0; i < 8 * (W - 1); ++i) hist[i] = 0;
  }
  const uint4 xin = *reinterpret_cast<const uint4*>(x + (long)n * x_pitch + d);
  float xv[W][8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
#pragma unroll
    for (int j = 0; j < W - 1; ++j) xv[j][c] = ix_bf2f(hist[c * (W - 1) + j]);
  }
  ix_unpack8(xin, xv[W - 1]);
  __attribute__((aligned(16))) bf16_t yv[8];
  ix_conv8_finish<W>(xv, wv, bias != nullptr, bv, silu, yv);
  if (row > 0) {
    // slide the window: slot j <- slot j + 1, last slot <- this step's input
    __attribute__((aligned(16))) bf16_t nh[8 * (W - 1)];
    const bf16_t* xb = reinterpret_cast<const bf16_t*>(&xin);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
      for (int j = 0; j < W - 2; ++j) nh[c * (W - 1) + j] = hist[c * (W - 1) + j + 1];
      nh[c * (W - 1) + W - 2] = xb[c];
    }
    uint4* o4 = reinterpret_cast<uint4*>(hp);
#pragma unroll
    for (int i = 0; i < 3; ++i) o4[i] = reinterpret_cast<const uint4*>(nh)[i];
  }
  bf16_t* yo = y + (long)n * D + d;
  if (d < qk_channels) {
    float v8[8], sq[8];
    ix_unpack8(*reinterpret_cast<const uint4*>(yv), v8);
#pragma unroll
    for (int i = 0; i < 8; ++i) sq[i] = v8[i] * v8[i];
    const float ssum = ix_lane_tree<16>(ix_tree8(sq));
    const float rn = ix_rsqrt_ieee(ssum + eps);
    __attribute__((aligned(16))) bf16_t out[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = ix_f2bf(v8[i] * rn);
    *reinterpret_cast<uint4*>(yo) = *reinterpret_cast<const uint4*>(out);
  } else {
    *reinterpret_cast<uint4*>(yo) = *reinterpret_cast<const uint4*>(yv);
  }
}

extern "C" int ix_gdn_decode_prep(const void* x, long x_pitch, const void* a, long a_pitch, const void* b, long b_pitch,
                                  const void* conv_weight, const void* conv_bias, const float* A_log,
                                  const float* dt_bias, void* conv_pool, const int* rows, void* y, float* g, void* beta,
                                  long N, long H, long K, long HV, long V, long W, int silu, float eps, void* stream) {
  if (!x || !a || !b || !conv_weight || !A_log || !dt_bias || !conv_pool || !rows || !y || !g || !beta) return IX_ERR_ARG;
  if (N < 0 || H <= 0 || K <= 0 || HV <= 0 || V <= 0) return IX_ERR_ARG;
  const long D = 2 * H * K + HV * V;
  if (x_pitch < D || a_pitch < HV || b_pitch < HV) return IX_ERR_ARG;
  // one head = 16 threads of eight channels; 16-byte accesses everywhere
  if (W != 4 || K != 128 || (D % 128) || (x_pitch % 8) || N > 65535) return IX_DECLINED;
  if (!ix_aligned(x, 16) || !ix_aligned(y, 16) || !ix_aligned(conv_weight, 16) || !ix_aligned(conv_pool, 16) ||
      (conv_bias && !ix_aligned(conv_bias, 16)))
    return IX_DECLINED;
  if (N == 0) return IX_OK;
  const long gx = (D / 8 + 255) / 256;
  hipLaunchKernelGGL(k_gdn_decode_prep, dim3((unsigned)gx, (unsigned)N), dim3(256), 0, (hipStream_t)stream,
                     (const bf16_t*)x, x_pitch, (const bf16_t*)a, a_pitch, (const bf16_t*)b, b_pitch,
                     (const bf16_t*)conv_weight, (const bf16_t*)conv_bias, A_log, dt_bias, (bf16_t*)conv_pool, rows,
                     (bf16_t*)y, g, (bf16_t*)beta, D, (int)(2 * H * K), (int)HV, silu, eps);
  return ix_launch_status();
}
