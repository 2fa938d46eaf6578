// One or two rows times a weight matrix with an activation in the epilogue: gemv.hip's kernel and plans, bf16 weights.
// The sums are not rounded ahead of the activation and its launch (2 us of a captured step) is gone.
#include <type_traits>

#include "gemv_kernel.h"

using namespace k8sllm;

extern "C" int k8s_gemv_rpw(int M, int N_out, int epi);
extern "C" int k8s_gemv_act_plan(int M, int N_out, int K, int pair, int* ks, int* splits, int* wgs, int* per);

// kind: gated 0, 1, 5 (W [2 N_out][K] = gate | up) or 7; partial: as k8s_gemv_plan asks for with epi 2 (gated) or 0.  -5: the
// switches or the size ask for a form of the GEMV that is not built here.
extern "C" int k8s_gemv_act(void* out, void* partial, const void* x, const void* W, int M, int N_out, int K, int kind,
                            float limit, float alpha, hipStream_t stream) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (M < 1 || M > 2 || K <= 0 || K % 8 != 0 || N_out <= 0 || (!pair && kind != 7)) return -1;
  int ks, splits, wgs, per;
  const int rc = k8s_gemv_act_plan(M, N_out, K, pair, &ks, &splits, &wgs, &per);
  if (rc != 0) return rc;
  if (splits > 1 && partial == nullptr) return -3;
  float* part = splits > 1 ? (float*)partial : nullptr;
  const int rpw = k8s_gemv_rpw(M, N_out, pair ? EPI_SWIGLU : EPI_BF16), half = pair ? N_out : 0;
  const dim3 grid(wgs, splits);
  const size_t lds = (size_t)M * ks * 2;
  const EpiAct act{kind, limit, alpha};
  auto go = [&](auto m, auto r) {
    constexpr int MM = decltype(m)::value, RR = decltype(r)::value;
    const auto* xx = (const bf16_t*)x;
#define GA(EE, LP) \
  gemv_kernel<MM, RR, EE, 0, false, 1, 256, false, LP><<<grid, 256, lds, stream>>>( \
      out, part, xx, W, N_out, K, ks, half, nullptr, nullptr, nullptr, 0.f, nullptr, GemvAr{}, act)
    if (pair) { if (per > 1) GA(EPI_GLU, true); else GA(EPI_GLU, false); }
    else { if (per > 1) GA(EPI_ELEM, true); else GA(EPI_ELEM, false); }
#undef GA
  };
  using std::integral_constant;
  if (M == 1) rpw == 2 ? go(integral_constant<int, 1>{}, integral_constant<int, 2>{}) : go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
  else rpw == 2 ? go(integral_constant<int, 2>{}, integral_constant<int, 2>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  if (splits > 1) {
    const int blocks = (M * N_out + 255) / 256;
    if (pair) gemv_finalize_kernel<EPI_GLU><<<blocks, 256, 0, stream>>>(out, part, M, N_out, splits, half, act);
    else gemv_finalize_kernel<EPI_ELEM><<<blocks, 256, 0, stream>>>(out, part, M, N_out, splits, half, act);
  }
  return (int)hipGetLastError();
}
