// K3/K8/K9/K11/K12 for SMALL decode batches (3..8 rows): out[M, N] = epi(x[M, K] . W[N, K]^T), the weights
// streamed from HBM exactly once (the decode GEMV of gemv.hip stages x in LDS, 64-128 KiB per
// workgroup at 4-8 rows, and re-stages it for every 8 output rows; mgemm's MFMA tiles waste 3/4 of a 16-row tile).
//
// Structure (one 256-thread workgroup = 4 waves; KW of them split K, 4 / KW row groups split the rows):
//  * every wave owns ONE k-slice of KPW elements for the whole launch and holds x[0..M)[slice] in registers
//    (CPL 16-byte chunks per lane per row: <= 128 VGPRs at 8 rows), loaded once -- no LDS staging, no per-row-set
//    re-staging, occupancy bound by registers only (2-3 workgroups per CU);
//  * the workgroup walks a band of output rows, NRT weight rows per step (one row set), the next set's loads
//    (non-temporal, 16 B per lane, 1 KiB contiguous per wave instruction) in flight while the current set is
//    consumed by v_dot2_f32_bf16 (bf16) or v_cvt_scalef32_pk_bf16_fp8 + v_dot2 (fp8 e4m3 with per-row scales);
//  * the NRT x M per-lane partial sums of a row set are reduced across the wave by a HALVING butterfly (each
//    xor step exchanges only the half of the values the lane gives away: NRT*M + 2 shuffles instead of 6 per
//    value), and one lane per value parks the wave's total in LDS;
//  * after the band, the KW k-slices are summed in a fixed order (deterministic), the RMS prologue's 1/rms (norm
//    gamma folded into W, statistics from the same x registers), the fp8 row scale and the epilogue (bf16, fp32
//    logits, SwiGLU of the [gate; up] halves, or the residual add in place) are applied and stored.
//  * K longer than one workgroup covers (KW x KPW) is split over G = gridDim.y workgroups: fp32 partial slabs and
//    sgemv_finalize_kernel (fixed order over the slices + epilogue).
#include "sgemv_kernel.h"

using namespace k8sllm;

namespace {
// Launch plan: (k elements per wave slice, waves per workgroup along K, k-groups).  Slices of 2048 elements
// (bf16: 4 chunks per lane = 128 x registers at 8 rows; fp8: 2) split 4 or 2 ways inside the workgroup, the
// split with less idle slice area wins (ties: more waves on K); K <= 1024 takes one 1024-element slice per wave and
// 4 row groups.
struct SgPlan {
  int kpw, kw, g;
};
SgPlan sg_plan(int K) {
  if (K <= 1024) return {1024, 1, 1};
  const int s = (K + 2047) / 2048;                   // 2048-element slices
  const int g4 = (s + 3) / 4, g2 = (s + 1) / 2;
  const int idle4 = g4 * 4 - s, idle2 = g2 * 2 - s;
  if (idle4 <= idle2) return {2048, 4, g4};
  return {2048, 2, g2};
}
}  // namespace

// Workspace floats for the partial slabs (0 when the plan has one k-group).
// The same plan k8s_sgemv takes for these operands (fp8: e4m3 weights), so the slabs always fit.
extern "C" long long k8s_sgemv_workspace(int M, int N, int K, int epi, int fp8) {
  SmPlan sp;
  const int g = sm_take(M, N, K, fp8 != 0, false, sp) ? sp.g : sg_plan(K).g;
  if (g <= 1) return 0;
  return (long long)g * M * (epi == SG_SWIGLU ? 2 : 1) * N;
}

static void sg_finalize(void* out, float* part, const bf16_t* rr, int M, int N, int G, int epi, bool has_res,
                        hipStream_t stream) {
  const int total = M * N, blocks = (total + 255) / 256;
  if (epi == SG_SWIGLU) sgemv_finalize_kernel<SG_SWIGLU, false><<<blocks, 256, 0, stream>>>(out, part, rr, M, N, G, EpiAct{});
  else if (epi == SG_F32) sgemv_finalize_kernel<SG_F32, false><<<blocks, 256, 0, stream>>>(out, part, rr, M, N, G, EpiAct{});
  else if (has_res) sgemv_finalize_kernel<SG_BF16, true><<<blocks, 256, 0, stream>>>(out, part, rr, M, N, G, EpiAct{});
  else sgemv_finalize_kernel<SG_BF16, false><<<blocks, 256, 0, stream>>>(out, part, rr, M, N, G, EpiAct{});
}

// out [M, N] (bf16, or fp32 for epi 1); x [M, K] bf16; W [N, K] (epi 2: [2N, K], gate rows then up rows) bf16, or
// e4m3 bytes when wscale != null (fp32 per weight row); res [M, N] bf16 for the residual epilogue (may be out);
// partial: k8s_sgemv_workspace floats.  norm: scale row m by 1/rms(x[m]) (the gamma folded into W).
// Returns 0, a negative argument error, or -5 when this kernel does not take the call (the caller routes it to
// mgemm).
extern "C" int k8s_sgemv(void* out, void* partial, const void* x, const void* W, const float* wscale, const void* res,
                         int M, int N, int K, int epi, int norm, float eps, hipStream_t stream) {
  if (M < 1 || M > 16 || N <= 0 || K <= 0) return -1;
  const bool fp8 = wscale != nullptr;
  if (K % (fp8 ? 16 : 8) != 0) return -1;
  if (epi < SG_BF16 || epi > SG_SWIGLU) return -1;
  const bool has_res = res != nullptr;
  if (has_res && (epi != SG_BF16 || norm)) return -5;
  const bf16_t* xx = (const bf16_t*)x;
  const bf16_t* rr = (const bf16_t*)res;
  SmPlan sp;
  if (sm_take(M, N, K, fp8, norm != 0, sp)) {
    if (norm && sp.g > 1) return -5;
    if (sp.g > 1 && partial == nullptr) return -3;
#define SMK(MT, JT, EE, NN, RR, F8) \
  g_last = sm_launch<MT, JT, EE, NN, RR, F8>(out, partial, xx, W, wscale, rr, M, N, K, eps, sp, stream)
#define SMK_COMBO(MT, JT, F8)                                                           \
  if (epi == SG_BF16 && norm) { SMK(MT, JT, SG_BF16, true, false, F8); }                \
  else if (epi == SG_BF16 && has_res) { SMK(MT, JT, SG_BF16, false, true, F8); }        \
  else if (epi == SG_BF16) { SMK(MT, JT, SG_BF16, false, false, F8); }                  \
  else if (epi == SG_SWIGLU && norm) { SMK(MT, JT, SG_SWIGLU, true, false, F8); }       \
  else if (epi == SG_SWIGLU) { SMK(MT, JT, SG_SWIGLU, false, false, F8); }              \
  else if (norm) { SMK(MT, JT, SG_F32, true, false, F8); }                              \
  else { SMK(MT, JT, SG_F32, false, false, F8); }
#define SMK_JT(MT)                                           \
  if (fp8) {   /* (sm_plan keeps fp8 at <= 4 steps) */      \
    if (sp.jt == 1) { SMK_COMBO(MT, 1, true) }               \
    else if (sp.jt == 2) { SMK_COMBO(MT, 2, true) }          \
    else { SMK_COMBO(MT, 4, true) }                          \
  } else if (sp.jt == 1) { SMK_COMBO(MT, 1, false) }         \
  else if (sp.jt == 2) { SMK_COMBO(MT, 2, false) }           \
  else if (sp.jt == 4) { SMK_COMBO(MT, 4, false) }           \
  else { SMK_COMBO(MT, 8, false) }
    bool g_last = false;   // (true: the launch reduces its k-groups itself)
    if (M <= 8) { SMK_JT(8) } else { SMK_JT(16) }
#undef SMK_JT
#undef SMK_COMBO
#undef SMK
    if (sp.g > 1 && !g_last) sg_finalize(out, (float*)partial, rr, M, N, sp.g, epi, has_res, stream);
    return (int)hipGetLastError();
  }
  if (M > 8) return -5;
  SgPlan p = sg_plan(K);
  if (norm && p.g > 1) return -5;
  if (p.g > 1 && partial == nullptr) return -3;
  // rows per workgroup: enough workgroups to put every CU to work (~512 per k-group, 2 per CU), at most SG_BAND;
  // fewer rows per wave re-read x (L2-resident) more often, so the band never drops below 4 rows
  const int nr = epi == SG_SWIGLU ? 1 : 2;
  int band = (N + 511) / 512;
  band = min(SG_BAND, max(4, (band + nr - 1) / nr * nr));
  const dim3 grid((N + band - 1) / band, p.g);
  const int half_rows = epi == SG_SWIGLU ? N : 0;
  float* part = p.g > 1 ? (float*)partial : nullptr;
#define SGL(MT, KPW, KW, EE, NN, RR, F8)                                                                     \
  sgemv_kernel<MT, KPW, KW, EE, NN, RR, F8><<<grid, 256, 0, stream>>>(out, part, xx, W, wscale, rr, M, N, K, \
                                                                       eps, half_rows, band)
#define SG_COMBO(MT, KPW, KW, F8)                                                           \
  if (epi == SG_BF16 && norm) { SGL(MT, KPW, KW, SG_BF16, true, false, F8); }               \
  else if (epi == SG_BF16 && has_res) { SGL(MT, KPW, KW, SG_BF16, false, true, F8); }       \
  else if (epi == SG_BF16) { SGL(MT, KPW, KW, SG_BF16, false, false, F8); }                 \
  else if (epi == SG_SWIGLU && norm) { SGL(MT, KPW, KW, SG_SWIGLU, true, false, F8); }      \
  else if (epi == SG_SWIGLU) { SGL(MT, KPW, KW, SG_SWIGLU, false, false, F8); }             \
  else if (norm) { SGL(MT, KPW, KW, SG_F32, true, false, F8); }                             \
  else { SGL(MT, KPW, KW, SG_F32, false, false, F8); }
#define SG_PLAN(MT, F8)                                           \
  if (p.kpw == 1024) { SG_COMBO(MT, 1024, 1, F8) }                \
  else if (p.kw == 4) { SG_COMBO(MT, 2048, 4, F8) }               \
  else { SG_COMBO(MT, 2048, 2, F8) }
  if (M <= 4) {
    if (fp8) { SG_PLAN(4, true) } else { SG_PLAN(4, false) }
  } else {
    if (fp8) { SG_PLAN(8, true) } else { SG_PLAN(8, false) }
  }
#undef SG_PLAN
#undef SG_COMBO
#undef SGL
  if (p.g > 1) sg_finalize(out, part, rr, M, N, p.g, epi, has_res, stream);
  return (int)hipGetLastError();
}
