// K3 / K8 / K9(+K10) / K11 / K12 at prefill row counts, bf16: the 4-wave big-tile MFMA GEMM (pgemm4_kernel.h, whose notes are there), its
// split-K combine and the entry points.
#include "pgemm4_kernel.h"

namespace k8sllm {

// Split-K combine: out[m, 4 q .. 4 q + 3] = epi(sum over slices of the slabs), slices in order.  One thread per
// 4 output features of one token; x scaling (RMS) and the residual as in the main kernel's epilogue.
// MXO (SwiGLU, fp8 weights): the output is MX e4m3 + E8M0 -- the 8 threads of a 32-feature block (adjacent, one
// wave) take the block's max by shuffles.  FP8 with xs == nullptr: MX activations (their scales were the MFMA's).
template <int EPI, bool RMS, bool FP8, bool MXO = false>
__global__ void __launch_bounds__(256) pgemm_reduce_kernel(void* __restrict__ out, const bf16_t* res,
                                                           const float* __restrict__ slab, int splits, int M,
                                                           int N_out, int half_rows, int wrows, int K, float eps,
                                                           const float* __restrict__ xs,
                                                           const float* __restrict__ wsc, uint8_t* __restrict__ oq,
                                                           uint8_t* __restrict__ oe) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const int qn = N_out / 4;
  if (idx >= (long long)M * qn) return;   // MXO: M * qn is a multiple of 8, so a block's 8 threads exit together
  const int m = (int)(idx / qn), n0 = (int)(idx - (long long)m * qn) * 4;
  const size_t stride = (size_t)M * wrows;
  f32x4 s = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < splits; ++k) {
    const float* p = slab + (size_t)k * stride + (size_t)m * wrows;
    s += *reinterpret_cast<const f32x4*>(p + n0);
    if (EPI == P4_SWIGLU) u += *reinterpret_cast<const f32x4*>(p + half_rows + n0);
  }
  float sx = 1.f;
  if (RMS) {
    float t = 0.f;
    for (int k = 0; k < splits; ++k) t += slab[(size_t)splits * stride + (size_t)k * M + m];
    sx = rsqrtf(t / (float)K + eps);
  }
  if (xs != nullptr) sx *= xs[m];   // fp8: the token's scale; bf16: 1 / rms of its row
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (EPI == P4_SWIGLU) {
      float gt = s[e] * sx, up = u[e] * sx;
      if (FP8) {
        gt *= wsc[n0 + e];
        up *= wsc[half_rows + n0 + e];
      }
      v[e] = p4_silu(gt) * up;
      if (MXO) v[e] = bf_round(v[e]);
    } else {
      v[e] = s[e] * sx * (FP8 ? wsc[n0 + e] : 1.f);
    }
  }
  if constexpr (MXO) {
    float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
    amax = lane_max<1>(amax);
    amax = lane_max<2>(amax);
    amax = lane_max<4>(amax);
    const uint32_t e = mx_e8m0(amax);
    *reinterpret_cast<uint32_t*>(oq + (size_t)m * N_out + n0) = mx_pack4(v[0], v[1], v[2], v[3], mx_inv_scale(e));
    if ((n0 & 31) == 0) oe[mx_scale_off(m, n0 >> 5, M)] = (uint8_t)e;
  } else if (EPI == P4_F32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + (size_t)m * N_out + n0) = f32x4{v[0], v[1], v[2], v[3]};
  } else {
    if (EPI == P4_BF16 && res != nullptr) {
      const p4_u32x2 rr = *reinterpret_cast<const p4_u32x2*>(res + (size_t)m * N_out + n0);
      v[0] += lo_bf(rr[0]);
      v[1] += hi_bf(rr[0]);
      v[2] += lo_bf(rr[1]);
      v[3] += hi_bf(rr[1]);
    }
    const p4_u32x2 o = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
    *reinterpret_cast<p4_u32x2*>(reinterpret_cast<bf16_t*>(out) + (size_t)m * N_out + n0) = o;
  }
}

// 1 / rms of every row of x [M][K] (K a multiple of 8, rows 16-byte aligned), a workgroup per row.
__global__ void __launch_bounds__(256) row_scale_kernel(float* __restrict__ out, const bf16_t* __restrict__ x, int K, float eps) {
  __shared__ float red[16];
  const u32x4* row = reinterpret_cast<const u32x4*>(x + (size_t)blockIdx.x * K);
  float s = 0.f;
#pragma unroll 4
  for (int i = threadIdx.x; i < K / 8; i += 256) {
    const u32x4 v = row[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) s += lo_bf(v[e]) * lo_bf(v[e]) + hi_bf(v[e]) * hi_bf(v[e]);
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) out[blockIdx.x] = rsqrtf(s / (float)K + eps);
}

}  // namespace k8sllm

using namespace k8sllm;

namespace {
template <int EPI, bool RMS, bool FP8, bool MXO = false>
int reduce_launch(void* out, const void* res, const float* slab, int splits, int M, int N_out, int half_rows,
                  int wrows, int K, float eps, const float* xs, const float* wsc, void* oq, void* oe, hipStream_t s) {
  const long long items = (long long)M * (N_out / 4);
  hipLaunchKernelGGL((pgemm_reduce_kernel<EPI, RMS, FP8, MXO>), dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                     s, out, static_cast<const bf16_t*>(res), slab, splits, M, N_out, half_rows, wrows, K, eps, xs,
                     wsc, static_cast<uint8_t*>(oq), static_cast<uint8_t*>(oe));
  return (int)hipGetLastError();
}
}  // namespace

// Split-K combine of pgemm slabs (also used by the fp8 kernel): slab = [splits][M][wrows] fp32, then (rms)
// [splits][M] row sums of squares.
extern "C" int k8s_pgemm_reduce(void* out, const void* res, const float* slab, int splits, int M, int N_out, int K,
                                int epi, int rms, float eps, const float* xs, const float* wsc, void* oq, void* oe,
                                hipStream_t s) {
  if (splits < 1 || M <= 0 || N_out <= 0 || N_out % 4) return -1;
  const int half = epi == P4_SWIGLU ? N_out : 0, wrows = epi == P4_SWIGLU ? 2 * N_out : N_out;
  const bool fp8 = wsc != nullptr;   // (xs == nullptr with fp8: MX activations)
  if (rms && fp8) return -6;
  if (oq != nullptr) {
    if (!fp8 || epi != P4_SWIGLU || oe == nullptr || N_out % 128) return -7;
    return reduce_launch<P4_SWIGLU, false, true, true>(out, res, slab, splits, M, N_out, half, wrows, K, eps, xs, wsc,
                                                      oq, oe, s);
  }
#define K8S_RED(E, R, F) \
  return reduce_launch<E, R, F>(out, res, slab, splits, M, N_out, half, wrows, K, eps, xs, wsc, nullptr, nullptr, s)
  if (fp8) {
    switch (epi) {
      case P4_BF16: K8S_RED(P4_BF16, false, true);
      case P4_F32: K8S_RED(P4_F32, false, true);
      case P4_SWIGLU: K8S_RED(P4_SWIGLU, false, true);
    }
  } else if (rms) {
    switch (epi) {
      case P4_BF16: K8S_RED(P4_BF16, true, false);
      case P4_F32: K8S_RED(P4_F32, true, false);
      case P4_SWIGLU: K8S_RED(P4_SWIGLU, true, false);
    }
  } else {
    switch (epi) {
      case P4_BF16: K8S_RED(P4_BF16, false, false);
      case P4_F32: K8S_RED(P4_F32, false, false);
      case P4_SWIGLU: K8S_RED(P4_SWIGLU, false, false);
    }
  }
#undef K8S_RED
  return -2;
}

namespace {
int p4_dense(const P4Args& a, int cfg, int epi, int norm, hipStream_t s) {
  return cfg < P4_TILES ? p4_cfg<0, P4_TILES>(a, cfg, epi, norm, s) : cfg < P4_WIDE ? p4_tiles(a, cfg, epi, norm, s)
                                                                                  : p4_wide(a, cfg, epi, norm, s);
}
int p4_act(const P4Args& a, int cfg, int kind, bool grouped, hipStream_t s) {
  if (cfg == 0) cfg = 4;                               // (the same tile)
  if (cfg >= P4_WIDE) return p4_wide_act(a, cfg, kind, grouped, s);
  if (cfg >= P4_TILES) return p4_tiles_act(a, cfg, kind, grouped, s);
  return grouped ? p4_act_cfg<true, 1, P4_TILES>(a, cfg, kind, s) : p4_act_cfg<false, 1, P4_TILES>(a, cfg, kind, s);
}
}  // namespace
P4Args p4_args(void* out, const void* x, const void* W, int M, int N_out, int K, bool pair, int cfg, int group_m, int groups = 0) {
  const int bp = 32 * p4_tile(cfg).fp, bq = 32 * p4_tile(cfg).fq, feat = pair ? bp / 2 : bp;
  P4Args a = {};
  a.out = out;
  a.x = static_cast<const uint8_t*>(x);
  a.W = static_cast<const uint8_t*>(W);
  a.kbytes = (uint32_t)K * 2u;
  a.M = M;
  a.N_out = N_out;
  a.half_rows = pair ? N_out : 0;
  a.wrows = pair ? 2 * N_out : N_out;
  a.K = K;
  a.m_tiles = (M + bq - 1) / bq;
  a.n_tiles = (N_out + feat - 1) / feat;
  a.ks = K / 32;
  a.splits = 1;
  a.group_m = group_m > 0 ? group_m : 1;
  a.nwg = a.m_tiles * a.n_tiles;
  a.groups = groups;
  a.spread = a.m_tiles == 1;
  p4_walk(a, cfg);
  a.wide = N_out % 8 == 0 && ((uintptr_t)out & 15) == 0;
  return a;
}

extern "C" int k8s_pgemm4_scaled(int cfg) { return cfg >= 0 && cfg < kP4NumCfgs && p4_scaled(cfg); }

extern "C" int k8s_pgemm4_num_configs() { return kP4NumCfgs; }

extern "C" int k8s_pgemm4_config(int cfg, int* bp, int* bq, int* lds_bytes) {
  if (cfg < 0 || cfg >= kP4NumCfgs) return -1;
  *bp = 32 * kP4Cfgs[cfg].fp;
  *bq = 32 * kP4Cfgs[cfg].fq;
  *lds_bytes = ((kP4Cfgs[cfg].dw + 1) * *bp + (kP4Cfgs[cfg].dx + 1) * *bq) * 128;
  return 0;
}

// Launch facts: workgroups and split-K slab elements (0 without split-K).
extern "C" int k8s_pgemm4_plan(int M, int N_out, int K, int epi, int cfg, int splits, int* nwg, long long* slab_elems) {
  if (cfg < 0 || cfg >= kP4NumCfgs || M <= 0 || N_out <= 0 || K <= 0 || splits < 1) return -1;
  if (K % 64 != 0 || N_out % 4 != 0) return -1;
  const int bp = 32 * kP4Cfgs[cfg].fp, bq = 32 * kP4Cfgs[cfg].fq;
  const int feat = epi == P4_SWIGLU ? bp / 2 : bp;
  const int ks = K / 32;
  if (splits > ks / 2) return -1;
  const long long tiles = (long long)((M + bq - 1) / bq) * ((N_out + feat - 1) / feat);
  if (tiles * splits > (1LL << 30)) return -1;
  const long long wrows = epi == P4_SWIGLU ? 2LL * N_out : N_out;
  *nwg = (int)(tiles * splits);
  *slab_elems = splits > 1 ? (long long)splits * M * wrows + (long long)splits * M : 0;
  return 0;
}

extern "C" int k8s_row_scale(float* out, const void* x, int M, int K, float eps, hipStream_t stream) {
  if (M < 0 || K <= 0 || K % 8 || ((uintptr_t)x & 15)) return -1;
  if (M == 0) return 0;
  hipLaunchKernelGGL(row_scale_kernel, dim3(M), dim3(256), 0, stream, out, static_cast<const bf16_t*>(x), K, eps);
  return (int)hipGetLastError();
}

// scale [M] fp32 (optional; bf16 and SwiGLU epilogues, tiles of k8s_pgemm4_scaled): 1 / rms of the rows of x, not from a prologue.
extern "C" int k8s_pgemm4(void* out, float* slab, const void* x, const void* W, int M, int N_out, int K, int epi,
                          int cfg, int splits, int group_m, const void* res, int rms, float eps, const float* scale,
                          hipStream_t stream) {
  int nwg;
  long long nsl;
  if (k8s_pgemm4_plan(M, N_out, K, epi, cfg, splits, &nwg, &nsl) != 0) return -1;
  if (splits > 1 && slab == nullptr) return -3;
  const long long kbytes = (long long)K * 2;
  const long long wrows = epi == P4_SWIGLU ? 2LL * N_out : (long long)N_out;
  if (wrows * kbytes >= (1LL << 32) || (long long)M * kbytes >= (1LL << 32)) return -5;   // 32-bit DMA offsets
  if (res != nullptr && epi != P4_BF16) return -6;
  const int bp = 32 * kP4Cfgs[cfg].fp, bq = 32 * kP4Cfgs[cfg].fq;
  const int feat = epi == P4_SWIGLU ? bp / 2 : bp;
  P4Args a = {};
  a.out = out;
  a.res = static_cast<const bf16_t*>(res);
  a.slab = slab;
  a.x = static_cast<const uint8_t*>(x);
  a.W = static_cast<const uint8_t*>(W);
  a.kbytes = (uint32_t)kbytes;
  a.M = M;
  a.N_out = N_out;
  a.half_rows = epi == P4_SWIGLU ? N_out : 0;
  a.wrows = (int)wrows;
  a.K = K;
  a.m_tiles = (M + bq - 1) / bq;
  a.n_tiles = (N_out + feat - 1) / feat;
  a.ks = K / 32;
  a.splits = splits;
  a.group_m = group_m > 0 ? group_m : 1;
  a.nwg = nwg;
  a.eps = eps;
  a.scale = scale;
  a.spread = a.m_tiles == 1;
  p4_walk(a, cfg);
  a.wide = res == nullptr && N_out % 8 == 0 && ((uintptr_t)out & 15) == 0;
  if (scale != nullptr && splits > 1) a.scale = nullptr;   // the sums of the slices are scaled by the combine
  int rc = p4_dense(a, cfg, epi, a.scale != nullptr ? P4_SCALED : scale == nullptr && rms ? P4_RMS : P4_PLAIN, stream);
  if (rc != 0 || splits == 1) return rc;
  return k8s_pgemm_reduce(out, res, slab, splits, M, N_out, K, epi, scale == nullptr && rms, eps, scale, nullptr, nullptr, nullptr,
                          stream);
}

// act(x W^T (+ bias)) in bf16: `kind` gated (0, 1, 5; W = [gate; up] rows, bias [2 N_out] optional) or 7 (elementwise).
extern "C" int k8s_pgemm4_act(void* out, const void* x, const void* W, int M, int N_out, int K, int cfg, int group_m, int kind,
                              float limit, float alpha, const void* bias, hipStream_t stream) {
  const bool pair = kind != 7;
  int nwg;
  long long nsl;
  if ((kind != 0 && kind != 1 && kind != 5 && kind != 7) || (!pair && bias != nullptr)) return -1;
  if (k8s_pgemm4_plan(M, N_out, K, pair ? P4_SWIGLU : P4_BF16, cfg, 1, &nwg, &nsl) != 0) return -1;
  const long long kbytes = (long long)K * 2;
  if ((pair ? 2LL : 1LL) * N_out * kbytes >= (1LL << 32) || (long long)M * kbytes >= (1LL << 32)) return -5;
  if (bias != nullptr && ((uintptr_t)bias & 7)) return -1;
  P4Args a = p4_args(out, x, W, M, N_out, K, pair, cfg, group_m);
  a.limit = limit;
  a.alpha = alpha;
  a.bias = static_cast<const bf16_t*>(bias);
  return p4_act(a, cfg, kind, false, stream);
}

// Grouped product over at most `rows` compact rows (x: M rows in memory, ldx elements apart): kind < 0 plain, or a gated kind
// with [groups][2 N_out][K] weights (last_limit: the last group's).
extern "C" int k8s_pgemm4_grouped(void* out, const void* x, const void* W, int M, int rows, int N_out, int K, int groups,
                                  const int* seg, const int* a_rows, long ldx, int cfg, int group_m, int kind, float limit,
                                  float alpha, float last_limit, hipStream_t stream) {
  const bool pair = kind >= 0;
  if (kind < -1 || (pair && kind > 1 && kind != 5)) return -1;
  if (rows <= 0) return 0;
  if (M <= 0 || N_out <= 0 || N_out % 4 || K <= 0 || K % 64 || groups <= 0 || (seg == nullptr && rows % groups) || cfg < 0 || cfg >= kP4Grouped) return -1;
  if (ldx < K || ldx % 8 || (((uintptr_t)x | (uintptr_t)W) & 15) || ((uintptr_t)out & 7)) return -1;
  const long long kbytes = (long long)K * 2, wrows = (pair ? 2LL : 1LL) * N_out;
  if (wrows * kbytes >= (1LL << 32) || (long long)M * ldx * 2 >= (1LL << 32)) return -5;   // 32-bit DMA offsets
  P4Args a = p4_args(out, x, W, rows, N_out, K, pair, cfg, group_m, groups);
  const int bq = 32 * p4_tile(cfg).fq;
  a.m_tiles = rows / bq + groups;        // whole tiles, and a partial one per group
  a.spread = groups >= 8 && rows <= 192LL * groups;
  a.fine = 0;
  p4_walk(a, cfg);
  if ((long long)a.m_tiles * a.n_tiles > (1LL << 30)) return -1;
  a.nwg = a.m_tiles * a.n_tiles;
  a.xbytes = (uint32_t)(ldx * 2);
  a.seg = seg;
  a.gsize = rows / groups;
  a.a_rows = a_rows;
  a.wstride = wrows * kbytes;
  a.limit = limit;
  a.alpha = alpha;
  a.last_limit = last_limit;
  return p4_act(a, cfg, kind, true, stream);
}
