// One decode step of the hybrid model as ONE call: the launches of every layer in order, from a table of the layers'
// device pointers that the caller fills anew for every step (nothing is remembered between calls) and one workspace.
//
// A step is a hundred launches of 3 - 30 us at small batches. Driven one by one from Python (an output allocation, a
// dozen attribute reads and a foreign call each) they cost 15 us apiece on the host, so that a step of one sequence took
// 1.7 ms of which the GPU worked 1.1; from here a launch is about 2 us. The launches themselves are the library's own
// entry points, so every value is computed by the code that computes it when the ops are called one at a time, plus three
// kernels that exist only here because they fold what the runtime does with tensor ops between the calls:
//   k_step_begin     slot -> row of every GatedDeltaNet layer with its use stamp (ix_gdn_resolve_rows, one launch per layer
//                    otherwise), the step's positions copied out of the context counters and checked, the packed offsets
//                    0..n
//   k_embed_rmsnorm  the embedding rows gathered into the residual stream and normalised, the context counters advanced
//   k_rope_append    q and k rotated (ix_rope_pairs8), k and v written to the caches at the step's positions
#include "ix_common.h"
#include "../../include/isoexec_hip.h"
#include <math.h>

#define IX_STEP_GDN_MAX 64  // GatedDeltaNet layers one k_step_begin launch resolves (kernel-argument space)

struct IxStepMap {
  const int64_t* slot2row;
  int64_t map_n;
  int64_t* last_used;
  int64_t* clock;
};
struct IxStepMaps {
  IxStepMap m[IX_STEP_GDN_MAX];
};

// What a sequence's next token is checked against: nothing behind this kernel knows an extent.
enum { IX_STEP_FITS = -1, IX_STEP_BAD_POSITION = 0, IX_STEP_BAD_TOKEN = 1 };  // the latter two: index into error[]
struct IxStepLimits {
  const int64_t* tokens;    // [n]
  int64_t vocab;
  const int* ctx;           // [n] the position of this token
  const int64_t* kv_start;  // [n] first cache token of the sequence
  int64_t cache_len;        // positions that the sequence's part of the cache and the rotary tables both hold
  int64_t cache_tokens;     // tokens of the whole cache
  __device__ __forceinline__ int check(int i) const {
    const int64_t p = ctx[i], start = kv_start[i], t = tokens[i];
    if (!(p >= 0 && p < cache_len && start >= 0 && start < cache_tokens && p < cache_tokens - start)) return IX_STEP_BAD_POSITION;
    return t >= 0 && t < vocab ? IX_STEP_FITS : IX_STEP_BAD_TOKEN;
  }
};

// Workgroup l < layers: layer l's rows; the last workgroup (pos not NULL): positions and offsets. A sequence whose position
// does not fit or whose token the embedding does not hold takes the step as a null lane -- row 0 of every state pool,
// position -1: no key and no state is stored, none is read, its output is NaN -- and is reported in error[0] or error[1]. The
// counters are advanced by a later launch (k_embed_rmsnorm), so every workgroup here checks the same values.
__global__ __launch_bounds__(256) void k_step_begin(IxStepMaps maps, int layers, const int64_t* __restrict__ slots, int n,
                                                    IxStepLimits lim, int* __restrict__ rows, int* __restrict__ pos,
                                                    int* __restrict__ cu, int* __restrict__ error) {
  const int l = blockIdx.x;
  if (l < layers) {
    const IxStepMap m = maps.m[l];
    const int64_t stamp = m.clock[0] + 1;
    for (int i = threadIdx.x; i < n; i += 256) {
      int64_t s = slots[i];
      s = s < 0 ? 0 : (s > m.map_n - 1 ? m.map_n - 1 : s);
      const int64_t r = lim.check(i) == IX_STEP_FITS ? m.slot2row[s] : 0;
      rows[(long)l * n + i] = (int)r;
      m.last_used[r] = stamp;
    }
    __syncthreads();
    if (threadIdx.x == 0) m.clock[0] = stamp;
    return;
  }
  if (!pos) return;
  for (int i = threadIdx.x; i <= n; i += 256) {
    cu[i] = i;
    if (i < n) {
      const int bad = lim.check(i);
      pos[i] = bad == IX_STEP_FITS ? lim.ctx[i] : -1;
      // host memory: seen by the host once the launch has ended, whatever the caller waits for
      if (bad != IX_STEP_FITS && error) __hip_atomic_store(error + bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// h[i] = table[tokens[i]], x[i] = norm(h[i]): the layout and sums of k_rmsnorm_reg<64, 0, NG> on the gathered row. A
// null lane (pos < 0: its token may lie outside the table) reads nothing and gives a row of NaNs. Advances ctx.
template <int NG>
__global__ __launch_bounds__(64) void k_embed_rmsnorm(const bf16_t* __restrict__ table,
                                                      const int64_t* __restrict__ tokens, const int* __restrict__ pos,
                                                      int* __restrict__ ctx, const bf16_t* __restrict__ w,
                                                      bf16_t* __restrict__ h, bf16_t* __restrict__ x, float eps,
                                                      int zero_centered) {
  constexpr int LPR = 64, N = LPR * 8 * NG;
  const int sub = threadIdx.x;
  const long row = blockIdx.x;
  const bool held = pos[row] >= 0;
  if (sub == 0) ctx[row] += 1;
  const bf16_t* src = table + (held ? tokens[row] : 0) * N + sub * 8;
  uint4 xp[NG], wp[NG];
#pragma unroll
  for (int c = 0; c < NG; ++c) xp[c] = *reinterpret_cast<const uint4*>(src + c * LPR * 8);
#pragma unroll
  for (int c = 0; c < NG; ++c) wp[c] = *reinterpret_cast<const uint4*>(w + sub * 8 + c * LPR * 8);
  float xv[NG][8];
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    if (!held) xp[c] = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
    *reinterpret_cast<uint4*>(h + row * N + sub * 8 + c * LPR * 8) = xp[c];
    ix_unpack8(xp[c], xv[c]);
    ix_sumsq8(xv[c], acc);
  }
  const float rstd = ix_norm_rstd<LPR>(acc, N, eps);
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    float wv[8], o[8];
    ix_unpack8(wp[c], wv);
    ix_norm8(xv[c], rstd, wv, zero_centered, o);
    ix_store8_bf16(x + row * N + sub * 8 + c * LPR * 8, 8, true, o);
  }
}

static bool ix_embed_rmsnorm_serves(long N) { return N == 512 || N == 1024 || N == 2048 || N == 4096; }

static int ix_embed_rmsnorm(const void* table, const int64_t* tokens, const int* pos, int* ctx, const void* w, void* h,
                            void* x, long n, long N, float eps, hipStream_t st) {
#define IX_EMB(NG_)                                                                                                     \
  if (N == 512 * NG_) {                                                                                                 \
    hipLaunchKernelGGL((k_embed_rmsnorm<NG_>), dim3((unsigned)n), dim3(64), 0, st, (const bf16_t*)table, tokens, \
                       pos, ctx, (const bf16_t*)w, (bf16_t*)h, (bf16_t*)x, eps, 1);                                     \
    return ix_launch_status();                                                                                          \
  }
  IX_EMB(1) IX_EMB(2) IX_EMB(4) IX_EMB(8)
#undef IX_EMB
  return IX_DECLINED;
}

// The projection row of a token holds HQ + HKV heads to rotate and HKV value heads, D each. Rotated q heads go back to the
// row, rotated k heads and the v heads to cache token kv_start[n] + pos[n] ([*, HKV, D]), which k_step_begin has checked
// against the cache and the tables; a null lane (pos < 0) stores neither. Eight pairs (or, for v, sixteen values) per
// thread; the rotation is ix_rope_pairs8, as in k_rope8.
__global__ __launch_bounds__(256) void k_rope_append(bf16_t* __restrict__ proj, long pitch, const bf16_t* __restrict__ cs,
                                                     const bf16_t* __restrict__ sn, const int* __restrict__ pos,
                                                     const int64_t* __restrict__ kv_start, bf16_t* __restrict__ kc,
                                                     bf16_t* __restrict__ vc, int HQ, int HKV, int D) {
  const int n = blockIdx.y;
  const int chunks = D >> 4;  // 8-pair chunks per head
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= (HQ + 2 * HKV) * chunks) return;
  const int c = i % chunks, hd = i / chunks, half = D >> 1;
  bf16_t* row = proj + (long)n * pitch + (long)hd * D + c * 8;
  const int p = pos[n];
  if (p < 0 && hd >= HQ) return;
  const uint4 a4 = *reinterpret_cast<const uint4*>(row), b4 = *reinterpret_cast<const uint4*>(row + half);
  const long slot = kv_start[n] + p;
  if (hd >= HQ + HKV) {
    bf16_t* d = vc + (slot * HKV + (hd - HQ - HKV)) * D + c * 8;
    *reinterpret_cast<uint4*>(d) = a4;
    *reinterpret_cast<uint4*>(d + half) = b4;
    return;
  }
  uint4 lo4, hi4;
  if (p < 0) {
    lo4 = hi4 = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
  } else {
    const bf16_t* ct = cs + (long)p * D + c * 8;
    const bf16_t* st = sn + (long)p * D + c * 8;
    const uint4 c0 = *reinterpret_cast<const uint4*>(ct), c1 = *reinterpret_cast<const uint4*>(ct + half);
    const uint4 s0 = *reinterpret_cast<const uint4*>(st), s1 = *reinterpret_cast<const uint4*>(st + half);
    ix_rope_pairs8(a4, b4, c0, c1, s0, s1, lo4, hi4);
  }
  bf16_t* d = hd < HQ ? row : kc + (slot * HKV + (hd - HQ)) * D + c * 8;
  *reinterpret_cast<uint4*>(d) = lo4;
  *reinterpret_cast<uint4*>(d + half) = hi4;
}

// ---- the step --------------------------------------------------------------------------------------------------------

namespace {

struct Carver {  // 256-byte aligned pieces of one workspace; with base NULL it only adds up
  char* base;
  size_t at = 0;
  explicit Carver(void* b) : base((char*)b) {}
  template <typename T>
  T* take(size_t count) {
    T* p = base ? reinterpret_cast<T*>(base + at) : nullptr;
    at += (count * sizeof(T) + 255) / 256 * 256;
    return p;
  }
};

struct Work {
  int *rows, *pos, *cu;
  bf16_t *h[2], *x, *proj, *mix, *y, *o, *yn, *inter, *eo;
  float *g, *logits, *prob, *pprob;
  bf16_t* beta;
  int *idx, *counts, *offsets, *sorted, *crows, *meta, *scratch;
  long max_tiles;
  int bm, bn;
  size_t bytes;
};

long proj_width(const IxDecodeDims& d, bool attention) {
  return attention ? (d.q_heads + 2 * d.kv_heads) * d.head_dim
                   : 2 * d.gdn_k_heads * d.gdn_head_dim + 2 * d.gdn_v_heads * d.gdn_head_dim + 2 * d.gdn_v_heads;
}

Work carve(const IxDecodeDims& d, void* base) {
  Work w;
  Carver c(base);
  const long n = d.n, E = d.experts, k = d.topk;
  const long gdn_d = 2 * d.gdn_k_heads * d.gdn_head_dim + d.gdn_v_heads * d.gdn_head_dim;
  const long pw = proj_width(d, false) > proj_width(d, true) ? proj_width(d, false) : proj_width(d, true);
  const long ow = d.gdn_v_heads * d.gdn_head_dim > d.q_heads * d.head_dim ? d.gdn_v_heads * d.gdn_head_dim
                                                                          : d.q_heads * d.head_dim;
  w.bm = d.packed_experts ? ix_moe_pick_bm_packed(n, k, E) : ix_moe_pick_bm(n, k, E);
  w.bn = w.bm == 128 ? 128 : 256;
  w.max_tiles = ix_moe_max_tiles(n, k, E, w.bm);
  w.rows = c.take<int>(n * d.layers);
  w.pos = c.take<int>(n);
  w.cu = c.take<int>(n + 1);
  w.h[0] = c.take<bf16_t>(n * d.hidden);
  w.h[1] = c.take<bf16_t>(n * d.hidden);
  w.x = c.take<bf16_t>(n * d.hidden);
  w.mix = c.take<bf16_t>(n * d.hidden);
  w.proj = c.take<bf16_t>(n * pw);
  w.y = c.take<bf16_t>(n * gdn_d);
  w.o = c.take<bf16_t>(n * ow);
  w.yn = c.take<bf16_t>(n * ow);
  w.g = c.take<float>(n * d.gdn_v_heads);
  w.beta = c.take<bf16_t>(n * d.gdn_v_heads);
  w.logits = c.take<float>(n * E);
  w.idx = c.take<int>(n * k);
  w.prob = c.take<float>(n * k);
  w.pprob = c.take<float>(n * k);
  w.counts = c.take<int>(E);
  w.offsets = c.take<int>(E + 1);
  w.sorted = c.take<int>(n * k);
  w.crows = c.take<int>(n * k);
  w.meta = c.take<int>(1 + 3 * w.max_tiles);
  w.scratch = c.take<int>(ix_moe_permute_scratch_ints(n, E) + 1);
  w.inter = c.take<bf16_t>(n * k * d.expert_inter);
  w.eo = c.take<bf16_t>(n * k * d.hidden);
  w.bytes = c.at;
  return w;
}

bool served(const IxDecodeDims& d) {
  if (d.n <= 0 || d.n > 65535 || d.layers <= 0 || d.vocab <= 0 || d.max_positions <= 0 || d.max_positions > 0x7fffffffL) return false;
  if (!ix_embed_rmsnorm_serves(d.hidden)) return false;
  // ix_moe_combine_add_rmsnorm's widths
  const long ng = d.hidden / 512;
  const bool comb = (d.topk == 8) || (d.topk == 4) || (d.topk == 2 && ng == 4);
  if (!comb) return false;
  if (d.gdn_head_dim != 128 || d.gdn_k_heads <= 0 || d.gdn_v_heads <= 0 || d.gdn_v_heads % d.gdn_k_heads) return false;
  if (d.head_dim != 128 || d.kv_heads <= 0 || d.q_heads % d.kv_heads || d.kv_heads > 65535) return false;
  const long grp = d.q_heads / d.kv_heads;
  if (grp > 32 || (grp & (grp - 1))) return false;
  if (d.experts <= 0 || d.experts > 512 || d.topk > d.experts || d.expert_inter <= 0 || d.expert_inter % 8) return false;
  return proj_width(d, false) % 8 == 0 && proj_width(d, true) % 8 == 0;
}

// Bytes a step moves at least, hence between two readings of one weight: every layer's projections, as many experts as the
// step can touch, the recurrent states read and written.
size_t step_bytes(const IxDecodeDims& d, const IxDecodeLayer* layers) {
  const long touched = d.n * d.topk < d.experts ? d.n * d.topk : d.experts;
  size_t sum = 0;
  for (long l = 0; l < d.layers; ++l) {
    const bool attention = layers[l].kind != 0;
    const long out = attention ? d.q_heads * d.head_dim : d.gdn_v_heads * d.gdn_head_dim;
    sum += (size_t)(proj_width(d, attention) + out + touched * 3 * d.expert_inter) * d.hidden * 2;
    if (!attention) sum += (size_t)d.n * d.gdn_v_heads * d.gdn_head_dim * d.gdn_head_dim * 8;
  }
  return sum;
}

}  // namespace

extern "C" size_t ix_decode_step_workspace_bytes(const IxDecodeDims* dims) {
  return dims && served(*dims) ? carve(*dims, nullptr).bytes : 0;
}

extern "C" int ix_decode_step_checked(const IxDecodeDims* dims, const IxDecodeCache* cache, const IxDecodeLayer* layers,
                                      const void* embed, const void* pre_norm, const void* cos_table, const void* sin_table,
                                      const int64_t* tokens, const int64_t* slots, int* ctx, const int64_t* kv_start,
                                      float eps, void* workspace, size_t workspace_bytes, void* out, void* stream) {
  if (!dims || !cache || !layers || !embed || !pre_norm || !cos_table || !sin_table || !tokens || !slots || !ctx ||
      !kv_start || !workspace || !out)
    return IX_ERR_ARG;
  const IxDecodeDims& d = *dims;
  if (!served(d) || cache->tokens <= 0 || cache->len <= 0) return IX_DECLINED;
  const Work w = carve(d, workspace);
  if (workspace_bytes < w.bytes || !ix_aligned(workspace, 256) || !ix_aligned(out, 16)) return IX_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  const long n = d.n, Hd = d.hidden;
  // From here a sub-call that does not return IX_OK ends the step with its code: `served` and the caller's checks (contiguous
  // 16-byte aligned operands) leave nothing for them to decline.
#define IX_STEP(call)            \
  {                              \
    const int rc_ = (call);      \
    if (rc_ != IX_OK) return rc_ > 0 ? IX_ERR_ARG : rc_; \
  }
  {
    const IxStepLimits lim{tokens, d.vocab, ctx, kv_start, cache->len < d.max_positions ? cache->len : d.max_positions,
                           cache->tokens};
    long l = 0;
    int row_base = 0;
    bool first = true;
    while (first || l < d.layers) {
      IxStepMaps maps;
      int cnt = 0;
      for (; l < d.layers && cnt < IX_STEP_GDN_MAX; ++l)
        if (layers[l].kind == 0)
          maps.m[cnt++] = IxStepMap{layers[l].slot2row, layers[l].map_n, layers[l].last_used, layers[l].clock};
      hipLaunchKernelGGL(k_step_begin, dim3((unsigned)(cnt + 1)), dim3(256), 0, st, maps, cnt, slots, (int)n, lim,
                         w.rows + (long)row_base * n, first ? w.pos : nullptr, w.cu, cache->error);
      row_base += cnt;
      first = false;
    }
    IX_STEP(ix_launch_status());
  }
  IX_STEP(ix_embed_rmsnorm(embed, tokens, w.pos, ctx, pre_norm, w.h[0], w.x, n, Hd, eps, st));
  const size_t footprint = step_bytes(d, layers);
  auto linear = [&](const bf16_t* a, long K, const void* weight, const void* packed, bf16_t* c, long N) -> int {
    if (packed && n <= 64) {
      const int rc = ix_gemm_bf16_nt_decode_footprint(a, K, packed, c, N, n, N, K, footprint, stream);
      if (rc != IX_DECLINED) return rc;
    }
    return ix_gemm_bf16_nt(a, K, weight, K, nullptr, c, IX_DT_BF16, N, n, N, K, 0, nullptr, 0, stream);
  };
  int gdn_seen = 0;
  for (long l = 0; l < d.layers; ++l) {
    const IxDecodeLayer& y = layers[l];
    bf16_t* h = w.h[0];
    if (y.kind == 0) {
      const long H = d.gdn_k_heads, HV = d.gdn_v_heads, K = d.gdn_head_dim;
      const long kd = H * K, D = 2 * kd + HV * K, pw = proj_width(d, false);
      const int* rows = w.rows + (long)(gdn_seen++) * n;
      IX_STEP(linear(w.x, Hd, y.w_in, y.w_in_packed, w.proj, pw));
      const bf16_t* z = w.proj + D;
      const bf16_t* b = z + HV * K;
      const bf16_t* a = b + HV;
      IX_STEP(ix_gdn_decode_prep(w.proj, pw, a, pw, b, pw, y.conv_weight, y.conv_bias, y.A_log, y.dt_bias, y.conv_state, rows,
                                 w.y, w.g, w.beta, n, H, K, HV, K, 4, 1, 1e-6f, stream));
      IX_STEP(ix_gdn_scan(w.y, w.y + kd, w.y + 2 * kd, w.g, w.beta, w.o, IX_DT_BF16, D, D, D, y.ssm_state, w.cu, rows, 0, n,
                          H, HV, K, K, (float)pow((double)K, -0.5), 1, stream));
      IX_STEP(ix_gated_out_norm(w.o, z, pw, y.out_norm, w.yn, n, HV, K, eps, 1, stream));
      IX_STEP(linear(w.yn, HV * K, y.w_out, y.w_out_packed, w.mix, Hd));
    } else {
      const long HQ = d.q_heads, HKV = d.kv_heads, D = d.head_dim, pw = proj_width(d, true);
      IX_STEP(linear(w.x, Hd, y.w_in, y.w_in_packed, w.proj, pw));
      const unsigned per = (unsigned)((HQ + 2 * HKV) * (D / 16));
      hipLaunchKernelGGL(k_rope_append, dim3((per + 255) / 256, (unsigned)n), dim3(256), 0, st, w.proj, pw,
                         (const bf16_t*)cos_table, (const bf16_t*)sin_table, w.pos, kv_start, (bf16_t*)y.k_cache,
                         (bf16_t*)y.v_cache, (int)HQ, (int)HKV, (int)D);
      IX_STEP(ix_launch_status());
      IX_STEP(ix_attn_varlen(w.proj, pw, y.k_cache, y.v_cache, HKV * D, w.o, w.cu, (const long*)kv_start, w.pos, n, 1, HQ,
                             HKV, D, (float)pow((double)D, -0.5), stream));
      IX_STEP(linear(w.o, HQ * D, y.w_out, y.w_out_packed, w.mix, Hd));
    }
    IX_STEP(ix_add_rmsnorm_gamma(w.mix, h, y.post_norm, w.x, w.h[1], n, Hd, eps, 1, stream));
    h = w.h[1];
    IX_STEP(ix_gemm_bf16_nt(w.x, Hd, y.router, Hd, nullptr, w.logits, IX_DT_F32, d.experts, n, d.experts, Hd, 0, nullptr, 0,
                            stream));
    if (n <= 256 && d.experts <= 128) {
      IX_STEP(ix_moe_route_one_tile(w.logits, d.experts, n, d.experts, d.topk, 1, 0.0f, w.bm, w.idx, w.prob, w.counts,
                                    w.offsets, w.sorted, w.pprob, w.crows, w.meta, w.max_tiles, stream));
    } else {
      IX_STEP(ix_moe_router_topk(w.logits, d.experts, n, d.experts, d.topk, 1, 0.0f, w.idx, w.prob, nullptr, nullptr, stream));
      IX_STEP(ix_moe_permute(w.idx, w.prob, n, d.experts, d.topk, w.bm, w.counts, w.offsets, w.sorted, w.pprob, w.crows,
                             w.meta, w.max_tiles, w.scratch, stream));
    }
    const bool streamed = d.packed_experts && (w.bm == 32 || w.bm == 64);
    if (streamed) {
      IX_STEP(ix_moe_experts_packed_footprint(w.x, Hd, w.sorted, w.pprob, y.w1_packed, y.w2_packed, w.meta, w.max_tiles,
                                              w.bm, w.inter, w.eo, n, n * d.topk, Hd, d.expert_inter, footprint, stream));
    } else {
      IX_STEP(ix_moe_experts_tile(w.x, Hd, w.sorted, w.pprob, y.w1, y.w2, w.meta, w.max_tiles, w.bm, w.bn, w.inter, w.eo, n,
                                  n * d.topk, Hd, d.expert_inter, stream));
    }
    void* x_out = l + 1 < d.layers ? (void*)w.x : out;
    IX_STEP(ix_moe_combine_add_rmsnorm(w.eo, w.crows, d.topk, (int)d.combine_fp32, h, y.next_norm, x_out, w.h[0], n, Hd, eps, 1,
                                       stream));
  }
#undef IX_STEP
  return IX_OK;
}

extern "C" int ix_decode_step(const IxDecodeDims* dims, const IxDecodeLayer* layers, const void* embed, const void* pre_norm,
                              const void* cos_table, const void* sin_table, const int64_t* tokens, const int64_t* slots,
                              int* ctx, const int64_t* kv_start, float eps, void* workspace, size_t workspace_bytes,
                              void* out, void* stream) {
  const IxDecodeCache unknown{INT64_MAX, INT64_MAX, nullptr};
  return ix_decode_step_checked(dims, &unknown, layers, embed, pre_norm, cos_table, sin_table, tokens, slots, ctx, kv_start,
                                eps, workspace, workspace_bytes, out, stream);
}
