// 3 - 16 rows times a weight matrix with an activation in the epilogue: sgemv.hip's MFMA kernel and plan, bf16 weights.
#include "sgemv_kernel.h"

using namespace k8sllm;

extern "C" long long k8s_sgemv_workspace(int M, int N, int K, int epi, int fp8);

// kind: gated 0, 1, 5 (W [2 N][K] = gate | up) or 7; partial: k8s_sgemv_workspace(M, N, K, 2 (gated) or 0, 0) floats.  -5: rows or
// a depth that the MFMA form does not take.
extern "C" int k8s_sgemv_act(void* out, void* partial, const void* x, const void* W, int M, int N, int K, int kind, float limit,
                             float alpha, hipStream_t stream) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (M < 1 || M > 16 || N <= 0 || K <= 0 || (!pair && kind != 7)) return -1;
  SmPlan sp;
  if (!sm_take(M, N, K, false, false, sp)) return -5;
  if (sp.g > 1 && partial == nullptr) return -3;
  const EpiAct act{kind, limit, alpha};
  bool whole = false;      // the launch reduces its k-groups itself
#define SA(MT, JT, EE) \
  whole = sm_launch<MT, JT, EE, false, false, false>(out, partial, (const bf16_t*)x, W, nullptr, nullptr, M, N, K, 0.f, sp, stream, act)
#define SA_JT(MT, EE)                  \
  if (sp.jt == 1) SA(MT, 1, EE);       \
  else if (sp.jt == 2) SA(MT, 2, EE);  \
  else if (sp.jt == 4) SA(MT, 4, EE);  \
  else SA(MT, 8, EE);
  if (pair) {
    if (M <= 8) { SA_JT(8, SG_GLU) } else { SA_JT(16, SG_GLU) }
  } else {
    if (M <= 8) { SA_JT(8, SG_ELEM) } else { SA_JT(16, SG_ELEM) }
  }
#undef SA_JT
#undef SA
  if (sp.g > 1 && !whole) {
    const int blocks = (M * N + 255) / 256;
    if (pair) sgemv_finalize_kernel<SG_GLU, false><<<blocks, 256, 0, stream>>>(out, (const float*)partial, nullptr, M, N, sp.g, act);
    else sgemv_finalize_kernel<SG_ELEM, false><<<blocks, 256, 0, stream>>>(out, (const float*)partial, nullptr, M, N, sp.g, act);
  }
  return (int)hipGetLastError();
}
