// K3/K8/K9/K11/K12 decode path: skinny GEMM out[M, N] = x[M, K] . W[N, K]^T for M <= 8 rows
// (decode batch), bf16 weights streamed from HBM exactly once.
//
// The weight stream is the whole cost (HBM-bound: 2 bytes per weight, ~1 FLOP/byte at M = 1),
// so the kernel is built around keeping many 16-byte weight loads in flight per lane:
//  * one wave owns RPW output rows; a workgroup = 4 waves shares one K-slice of x staged in
//    LDS (x is re-read by every row, the LDS read is 256 B/clk/CU vs the L1's 64),
//  * weights are loaded with non-temporal hints (read once: keep them out of L2/MALL),
//  * bf16 pairs are multiplied with v_dot2_f32_bf16 (fp32 accumulate),
//  * when N alone gives too few workgroups to fill 256 CUs, K is split (grid.y) and partial
//    fp32 slabs are combined by a finalize kernel that also applies the epilogue;
//  * for small N (e.g. the TP = 8 QKV / gate-up slices) KW waves of a workgroup share one row
//    set and split its K range (reduced through LDS), so every wave's share of the weight
//    stream is in flight at once instead of taking several dependent rounds.
// Epilogues: BF16 store, FP32 store (logits), SWIGLU: W = [gate; up] (2I rows) and the output is
// silu(gate_j) * up_j (SURVEY.md K10 fused into K9).
// FP8 weights: W holds OCP e4m3 bytes with one fp32 scale per row; a 16-byte
// load carries 16 weights (half the HBM bytes of bf16); every dword of four e4m3 is converted to two
// bf16 pairs with v_cvt_scalef32_pk_bf16_fp8 (exact) and fed to v_dot2_f32_bf16 against the packed
// activations; the row scale is applied once in the epilogue.
#include <cstdlib>

#include "gemv_kernel.h"

using namespace k8sllm;

// Plan the launch: returns the K-slice length (multiple of 512) and the split count.
// Rows per wave: 2 from M = 4 on.  Below, the plain (no norm prologue, no SwiGLU) projections with
// N >= 8192 outputs (o_proj, down at every TP degree) also take 2: half as many workgroups, twice the
// weight loads in flight per lane (measured TP = 8: o_proj 4.8 -> 3.6 us, down 10.8 -> 9.9 us; it
// loses on the small-N QKV and on gate/up, profiles/kbench_*).  K8S_GEMV_RPW1 = 1 / 2 forces M < 4.
static int gemv_rpw(int M, int N_out = 0, int epi = 0, int mode = 0) {
  static const int env = [] { const char* e = getenv("K8S_GEMV_RPW1"); return e ? atoi(e) : 0; }();
  if (M >= 4) return 2;
  if (env == 1 || env == 2) return env;
  return (mode == 0 && epi != EPI_SWIGLU && N_out >= 8192) ? 2 : 1;
}

extern "C" int k8s_gemv_rpw(int M, int N_out, int epi) { return gemv_rpw(M, N_out, epi, 0); }

extern "C" void k8s_gemv_plan(int M, int N_out, int K, int epi, int mode, int* ks_out, int* splits_out) {
  const int rpw = gemv_rpw(M, N_out, epi, mode);
  const int rows_per_wg = 4 * rpw;
  const int n_wg = (N_out + rows_per_wg - 1) / rows_per_wg;
  const int lds_cap_elems = 65536 / (2 * M);  // <= 64 KiB of x per workgroup (M=1: K up to 32768 unsplit)
  int splits = 1;
  const int target = 256;  // split K only when N alone cannot give every CU a workgroup
  if (n_wg < target) splits = (target + n_wg - 1) / n_wg;
  int ks = (K + splits - 1) / splits;
  ks = ((ks + 511) / 512) * 512;
  if (ks < 512) ks = 512;
  while (ks > lds_cap_elems) ks -= 512;
  if (ks > K) ks = ((K + 7) / 8) * 8;
  splits = (K + ks - 1) / ks;
  (void)epi;
  *ks_out = ks;
  *splits_out = splits;
}

// partial: fp32 workspace of splits * M * wrows floats (wrows = N_out, or 2*N_out for SWIGLU);
// may be null when the plan has a single split.
// wscale != null: W is fp8 (OCP e4m3, one fp32 scale per weight row); K must be a multiple of 16.
// mode: 0 plain, 1 norm weight nw applied in the prologue, 2 norm weight folded into W (nw unused)
// Row-set loop (LOOP): workgroups per CU the grid is cut to (0 = one row set per wave; -1 = default: 2 for fp8
// weights; for bf16 weights 2 on the plain bf16 epilogue (QKV, O, down) and off for SwiGLU / fp32 (gate/up, LM
// head)).  Measured on the 70B decode (profiles/gemv_loop_probe_r3.txt, bench A/B in
// profiles/bench_r3_gemv_loop_ab.txt): fp8 decode -0.6 %; bf16 with the loop everywhere +1.3 % (slower), on the
// plain-epilogue projections only -0.3 %.
// K8S_GEMV_LOOP sets it at load; k8s_gemv_set_loop changes it (tests, A/B probes).
static int g_gemv_loop = [] { const char* e = getenv("K8S_GEMV_LOOP"); return e ? atoi(e) : -1; }();
static int g_gemv_wide = [] { const char* e = getenv("K8S_GEMV_WIDE"); return e ? atoi(e) : 1; }();
extern "C" int k8s_gemv_set_wide(int on) {
  const int old = g_gemv_wide;
  if (on >= 0) g_gemv_wide = on;
  return old;
}
// bf16 SwiGLU (gate/up) GEMVs take the loop (2 workgroups per CU) when their one-row-set grid has at most this many
// workgroups: TP = 4 / 8 shapes (K8S_GEMV_LOOP_SWIGLU_MAX).  At one TP = 8 rank's shapes decode 4.554 -> 4.466
// ms/token (profiles/bench_r3_gemv_loop_ab.txt); at TP = 1 (7168 workgroups) the loop measured slower.
static int g_gemv_loop_swiglu_max = [] {
  const char* e = getenv("K8S_GEMV_LOOP_SWIGLU_MAX");
  return e ? atoi(e) : 2048;
}();
// smallest matrix (Mi weights) the fp8 / plain-epilogue loop takes (K8S_GEMV_LOOP_MIN_MI): 65 keeps the 70B O
// projection (exactly 64 Mi) off it -- +1.3 % end to end (profiles/bench_r3_gemv_loop_ab.txt)
static int g_gemv_loop_min_mi = [] { const char* e = getenv("K8S_GEMV_LOOP_MIN_MI"); return e ? atoi(e) : 65; }();
// default for bf16 weights with the plain bf16 epilogue (QKV, O, down -- not gate/up nor the LM head)
static int g_gemv_loop_bf16 = [] { const char* e = getenv("K8S_GEMV_LOOP_BF16"); return e ? atoi(e) : 2; }();
extern "C" int k8s_gemv_set_loop(int wg_per_cu) {   // returns the previous setting; < -1 only reads it
  const int old = g_gemv_loop;
  if (wg_per_cu >= -1) g_gemv_loop = wg_per_cu;
  return old;
}

// KW: waves per row set (K8S_GEMV_KW = 2 / 4 splits a row set's K over that many waves).  One wave per row
// set is the default: the two-wave split the small-N projections (TP = 8 QKV, LM head) used to take measured
// slower end to end (TP = 8 shapes 4.28 -> 4.26 ms/token with one wave, 8B and TP = 1 unchanged,
// profiles/gemv_kw_ab.txt).
static int gemv_kw() {
  static const int env = [] { const char* e = getenv("K8S_GEMV_KW"); return e ? atoi(e) : 0; }();
  return (env == 2 || env == 4) ? env : 1;
}
// Workgroups per CU of the row-set loop over a grid of `wgs` one-row-set workgroups; 0: no loop.
static int gemv_loop_wg(bool fp8, int M, int N_out, int K, int epi, int mode, int splits, int wgs) {
  const bool swiglu_loop = epi == EPI_SWIGLU && wgs <= g_gemv_loop_swiglu_max;
  // the loop only on matrices of >= 64 Mi weights (the 70B's at TP = 1, gate/up at TP = 4): on the smaller ones
  // (Llama-3-8B, fp8 at TP = 4) it measured slower
  const bool big = (long long)(epi == EPI_SWIGLU ? 2 * N_out : N_out) * K >= ((long long)g_gemv_loop_min_mi << 20);
  const bool plain_loop = epi == EPI_BF16 && big;
  const int wg = g_gemv_loop >= 0 ? g_gemv_loop
                                  : (fp8 ? (big ? 2 : 0) : (plain_loop ? g_gemv_loop_bf16 : (swiglu_loop ? 2 : 0)));
  return wg > 0 && splits == 1 && gemv_kw() == 1 && mode != 1 && M <= 2 && wgs > 256 * wg ? wg : 0;
}
// wide: 8-wave workgroups for the looped plain bf16-epilogue projections whose x slice takes >= 32 KiB of LDS (the
// down projection, K = 28672: 56 KiB): LDS, not waves, bounds those at 2 workgroups per CU, so twice the waves
// per workgroup put twice the weight loads in flight per CU (K8S_GEMV_WIDE = 0 turns it off)
static bool gemv_is_wide(int M, int K, int epi, int mode) {
  return g_gemv_wide && mode == 0 && epi == EPI_BF16 && (long long)M * K * 2 >= 32768;
}

// The launch of gemv_act.hip's products, the one that k8s_gemv makes of epi 2 (gated) or 0 (elementwise) under the same switches:
// k slice, splits, workgroups and (per > 1) row sets a wave.  -5: a form that is not built there.
extern "C" int k8s_gemv_act_plan(int M, int N_out, int K, int pair, int* ks, int* splits, int* wgs, int* per) {
  const int epi = pair ? EPI_SWIGLU : EPI_BF16;
  k8s_gemv_plan(M, N_out, K, epi, 0, ks, splits);
  const int rows = 4 * gemv_rpw(M, N_out, epi, 0), one = (N_out + rows - 1) / rows;
  const int wg = gemv_loop_wg(false, M, N_out, K, epi, 0, *splits, one);
  if (gemv_kw() != 1 || (wg > 0 && gemv_is_wide(M, K, epi, 0))) return -5;
  *per = wg > 0 ? (one + 256 * wg - 1) / (256 * wg) : 1;
  *wgs = (one + *per - 1) / *per;
  return 0;
}

static int gemv_launch(int mode, void* out, void* partial, const void* x, const void* W, const float* wscale, int M,
                       int N_out, int K, int epi, const void* res_in, void* res_out, const void* nw, float eps,
                       hipStream_t stream) {
  if (M < 1 || M > 8 || K % 8 != 0 || N_out <= 0) return -1;
  const bool fp8 = wscale != nullptr;
  if (fp8 && K % 16 != 0) return -1;
  int ks, splits;
  k8s_gemv_plan(M, N_out, K, epi, mode, &ks, &splits);
  if (splits > 1 && partial == nullptr) return -3;
  float* part = splits > 1 ? (float*)partial : nullptr;
  const int rpw = gemv_rpw(M, N_out, epi, mode);
  const int kw = gemv_kw();
  // The norm variants keep 4 row sets per workgroup when they split K (8 waves, 512 threads):
  // the per-workgroup norm prologue is then shared by twice the waves instead of being repeated.
  const int nt = (mode != 0 && kw == 2 && M <= 4) ? 512 : 256;
  const int rows_per_wg = (nt / 64 / kw) * rpw;
  dim3 grid((N_out + rows_per_wg - 1) / rows_per_wg, splits);
  const size_t lds = (size_t)M * ks * 2;
  const int half_rows = (epi == EPI_SWIGLU) ? N_out : 0;
  const bf16_t* xx = (const bf16_t*)x;
  const void* ww = W;
  const bf16_t* ri = (const bf16_t*)res_in;
  bf16_t* ro = (bf16_t*)res_out;
  const bf16_t* gw = (const bf16_t*)nw;
  const int loop_wg = gemv_loop_wg(fp8, M, N_out, K, epi, mode, splits, (int)grid.x);
  if (loop_wg > 0) {
    const bool wide = gemv_is_wide(M, K, epi, mode);
    if (wide) {
      const int wgs = (N_out + 8 * rpw - 1) / (8 * rpw);
      {
        const int per = (wgs + 256 * loop_wg - 1) / (256 * loop_wg);   // >= 1
        const dim3 wgrid((wgs + per - 1) / per, 1);
#define GW(MM, RR, F8)                                                                                              \
  gemv_kernel<MM, RR, EPI_BF16, 0, F8, 1, 512, false, true><<<wgrid, 512, lds, stream>>>(                           \
      out, nullptr, xx, ww, N_out, K, ks, half_rows, ri, ro, gw, eps, wscale, GemvAr{}, EpiAct{})
#define GW2(MM, RR) \
  if (fp8) { GW(MM, RR, true); } else { GW(MM, RR, false); }
        if (M == 1) { if (rpw == 2) { GW2(1, 2) } else { GW2(1, 1) } }
        else { if (rpw == 2) { GW2(2, 2) } else { GW2(2, 1) } }
#undef GW2
#undef GW
        return (int)hipGetLastError();
      }
    }
    const int per = ((int)grid.x + 256 * loop_wg - 1) / (256 * loop_wg);   // row sets per wave
    const dim3 lgrid(((int)grid.x + per - 1) / per, 1);
#define GL(MM, RR, EE, F8, NN)                                                                                     \
  gemv_kernel<MM, RR, EE, NN, F8, 1, 256, false, true><<<lgrid, 256, lds, stream>>>(out, nullptr, xx, ww, N_out, K, \
                                                                                     ks, half_rows, ri, ro, gw, eps, \
                                                                                     wscale, GemvAr{}, EpiAct{})
#define GL2(MM, RR, EE)                                             \
  if (fp8) { if (mode == 2) { GL(MM, RR, EE, true, 2); } else { GL(MM, RR, EE, true, 0); } }    \
  else { if (mode == 2) { GL(MM, RR, EE, false, 2); } else { GL(MM, RR, EE, false, 0); } }
#define GLE(MM, RR)                                      \
  switch (epi) {                                         \
    case EPI_BF16: GL2(MM, RR, EPI_BF16); break;         \
    case EPI_F32: GL2(MM, RR, EPI_F32); break;           \
    case EPI_SWIGLU: GL2(MM, RR, EPI_SWIGLU); break;     \
    default: return -2;                                  \
  }
    if (M == 1) { if (rpw == 2) { GLE(1, 2) } else { GLE(1, 1) } }
    else { if (rpw == 2) { GLE(2, 2) } else { GLE(2, 1) } }
#undef GLE
#undef GL2
#undef GL
    return (int)hipGetLastError();
  }
#define G4(MM, RR, EE, F8, KK, NTT)                                                                            \
  if (mode == 1) gemv_kernel<MM, RR, EE, 1, F8, KK, NTT><<<grid, NTT, lds, stream>>>(                          \
      out, part, xx, ww, N_out, K, ks, half_rows, ri, ro, gw, eps, wscale, GemvAr{}, EpiAct{});                            \
  else if (mode == 2) gemv_kernel<MM, RR, EE, 2, F8, KK, NTT><<<grid, NTT, lds, stream>>>(                     \
      out, part, xx, ww, N_out, K, ks, half_rows, ri, ro, gw, eps, wscale, GemvAr{}, EpiAct{});                            \
  else gemv_kernel<MM, RR, EE, 0, F8, KK><<<grid, 256, lds, stream>>>(out, part, xx, ww, N_out, K, ks,          \
                                                                       half_rows, ri, ro, gw, eps, wscale, GemvAr{}, EpiAct{})
#define G3(MM, RR, EE, F8, KK)                  \
  if constexpr (KK == 2 && MM <= 4) {           \
    G4(MM, RR, EE, F8, KK, 512);                \
  } else {                                      \
    G4(MM, RR, EE, F8, KK, 256);                \
  }
#define G2(MM, RR, EE, F8)                      \
  if (kw == 4) { G3(MM, RR, EE, F8, 4); }        \
  else if (kw == 2) { G3(MM, RR, EE, F8, 2); }   \
  else { G3(MM, RR, EE, F8, 1); }
#define G(MM, RR, EE)        \
  if (fp8) { G2(MM, RR, EE, true); } \
  else { G2(MM, RR, EE, false); }
#define BY_EPI(MM, RR)                  \
  switch (epi) {                        \
    case EPI_BF16: G(MM, RR, EPI_BF16); break;       \
    case EPI_F32: G(MM, RR, EPI_F32); break;         \
    case EPI_SWIGLU: G(MM, RR, EPI_SWIGLU); break;   \
    default: return -2;                 \
  }
  switch (M) {
    case 1: if (rpw == 2) { BY_EPI(1, 2) } else { BY_EPI(1, 1) } break;
    case 2: if (rpw == 2) { BY_EPI(2, 2) } else { BY_EPI(2, 1) } break;
    case 3: if (rpw == 2) { BY_EPI(3, 2) } else { BY_EPI(3, 1) } break;
    case 4: BY_EPI(4, 2) break;
    case 5: BY_EPI(5, 2) break;
    case 6: BY_EPI(6, 2) break;
    case 7: BY_EPI(7, 2) break;
    case 8: BY_EPI(8, 2) break;
  }
#undef BY_EPI
#undef G
#undef G2
#undef G3
  if (splits > 1) {
    const int total = M * N_out;
    const int blocks = (total + 255) / 256;
    switch (epi) {
      case EPI_BF16: gemv_finalize_kernel<EPI_BF16><<<blocks, 256, 0, stream>>>(out, part, M, N_out, splits, half_rows, EpiAct{}); break;
      case EPI_F32: gemv_finalize_kernel<EPI_F32><<<blocks, 256, 0, stream>>>(out, part, M, N_out, splits, half_rows, EpiAct{}); break;
      case EPI_SWIGLU: gemv_finalize_kernel<EPI_SWIGLU><<<blocks, 256, 0, stream>>>(out, part, M, N_out, splits, half_rows, EpiAct{}); break;
    }
  }
  return (int)hipGetLastError();
}

extern "C" int k8s_gemv_norm_w(void* out, void* partial, const void* x, const void* W, const float* wscale, int M,
                               int N_out, int K, int epi, const void* res_in, void* res_out, const void* nw,
                               float eps, hipStream_t stream) {
  return gemv_launch(nw != nullptr ? 1 : 0, out, partial, x, W, wscale, M, N_out, K, epi, res_in, res_out, nw, eps,
                     stream);
}

// Pre-norm projection with the norm weight folded into W: y = epi((W' . (x + res_in)) / rms(x + res_in)).
extern "C" int k8s_gemv_rms(void* out, void* partial, const void* x, const void* W, const float* wscale, int M,
                            int N_out, int K, int epi, const void* res_in, void* res_out, float eps,
                            hipStream_t stream) {
  return gemv_launch(2, out, partial, x, W, wscale, M, N_out, K, epi, res_in, res_out, nullptr, eps, stream);
}

extern "C" int k8s_gemv_norm(void* out, void* partial, const void* x, const void* W, int M, int N_out, int K,
                             int epi, const void* res_in, void* res_out, const void* nw, float eps,
                             hipStream_t stream) {
  return k8s_gemv_norm_w(out, partial, x, W, nullptr, M, N_out, K, epi, res_in, res_out, nw, eps, stream);
}

extern "C" int k8s_gemv(void* out, void* partial, const void* x, const void* W, int M, int N_out, int K, int epi,
                        hipStream_t stream) {
  return k8s_gemv_norm_w(out, partial, x, W, nullptr, M, N_out, K, epi, nullptr, nullptr, nullptr, 0.f, stream);
}

extern "C" int k8s_gemv_fp8(void* out, void* partial, const void* x, const void* W, const float* wscale, int M,
                            int N_out, int K, int epi, const void* res_in, void* res_out, const void* nw, float eps,
                            hipStream_t stream) {
  if (wscale == nullptr) return -1;
  return k8s_gemv_norm_w(out, partial, x, W, wscale, M, N_out, K, epi, res_in, res_out, nw, eps, stream);
}

// Row-parallel projection with the tensor-parallel all-reduce (and the residual add) in its epilogue:
// out[M, N_out] = residual + sum over ranks of x . W^T (see GemvAr).  Every rank must issue the same sequence of
// these calls with the same shapes (the group epochs advance per call).  Two-row waves, one K slice (the whole
// row of x in LDS), 4-wave workgroups.  Returns -5 where the shape does not fit that plan (the caller then runs
// the GEMV and a separate all-reduce).
extern "C" int k8s_gemv_allreduce(void* out, const void* x, const void* W, const float* wscale, int M, int N_out,
                                  int K, const void* residual, void* const* bases, long long row_bytes,
                                  uint32_t* epochs, uint32_t* tickets, uint32_t* err, int rank, int world,
                                  long long timeout_ticks, hipStream_t stream) {
  constexpr int ROWS_WG = 8;  // 4 waves x 2 rows
  if (M < 1 || M > 8 || K % 16 != 0 || N_out <= 0 || world < 2 || world > GAR_MAX_WORLD || rank < 0 || rank >= world)
    return -1;
  if (N_out % ROWS_WG != 0 || (long long)M * K * 2 > 65536 || (long long)M * N_out * 4 > row_bytes) return -5;
  // row-set loop (K8S_GEMV_LOOP_AR = workgroups per CU, 0 = one row set per wave): each workgroup streams a
  // contiguous band of row sets and pushes each set's words as it finishes it
  static const int loop_ar = [] { const char* e = getenv("K8S_GEMV_LOOP_AR"); return e ? atoi(e) : 0; }();
  const int nwg1 = N_out / ROWS_WG;
  const int per = (loop_ar > 0 && M <= 2 && nwg1 > 256 * loop_ar) ? (nwg1 + 256 * loop_ar - 1) / (256 * loop_ar) : 1;
  const int nwg = (nwg1 + per - 1) / per;
  const int group = (nwg + 31) / 32;  // ~32 arrival groups: one waiting workgroup per group
  if ((nwg + group - 1) / group > GAR_MAX_GROUPS) return -5;
  GemvAr a;
  for (int i = 0; i < GAR_MAX_WORLD; ++i) a.base[i] = i < world ? static_cast<char*>(bases[i]) : nullptr;
  a.row_bytes = row_bytes; a.epochs = epochs; a.tickets = tickets; a.err = err;
  a.res = static_cast<const bf16_t*>(residual); a.timeout_ticks = timeout_ticks;
  a.rank = rank; a.world = world; a.group = group;
  const bool fp8 = wscale != nullptr;
  const size_t lds = (size_t)M * K * 2;
  const bf16_t* xx = static_cast<const bf16_t*>(x);
#define GAR1(MM, LP)                                                                                                \
  if (fp8) gemv_kernel<MM, 2, EPI_BF16, 0, true, 1, 256, true, LP><<<nwg, 256, lds, stream>>>(                      \
      out, nullptr, xx, W, N_out, K, K, 0, nullptr, nullptr, nullptr, 0.f, wscale, a, EpiAct{});                               \
  else gemv_kernel<MM, 2, EPI_BF16, 0, false, 1, 256, true, LP><<<nwg, 256, lds, stream>>>(                         \
      out, nullptr, xx, W, N_out, K, K, 0, nullptr, nullptr, nullptr, 0.f, wscale, a, EpiAct{})
#define GAR(MM)                                   \
  if constexpr (MM <= 2) {                        \
    if (per > 1) { GAR1(MM, true); }              \
    else { GAR1(MM, false); }                     \
  } else {                                        \
    GAR1(MM, false);                              \
  }
  switch (M) {
    case 1: GAR(1); break;
    case 2: GAR(2); break;
    case 3: GAR(3); break;
    case 4: GAR(4); break;
    case 5: GAR(5); break;
    case 6: GAR(6); break;
    case 7: GAR(7); break;
    case 8: GAR(8); break;
  }
#undef GAR
#undef GAR1
  return (int)hipGetLastError();
}

extern "C" int k8s_gemv_allreduce_max_groups() { return GAR_MAX_GROUPS; }
