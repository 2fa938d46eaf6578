// Decoding 1 - 16 rows of a model with an fp32 residual stream, the norms of a layer without launches of their own: the product that
// ends a sublayer (N: the stream's width) adds to the stream and leaves, next to it, the rows times the next norm's weight in bf16 and
// every workgroup's sums of squares; the product that begins the next sublayer (K: the width) takes those rows as its input and adds
// up the sums while its first weights are on their way.  A norm is one factor a row, so the product's fp32 sums take it as well as its
// input does -- the rows are rounded to bf16 once, as they were with the factor in them, and the branch is not rounded at all.
// sgemv.hip's MFMA kernel (sgemv_kernel.h) at every row count.  Bound by the weights' way from memory and, below some 10 MB, by the
// start of a launch.  us, product + norm + product / here, weights from memory: 8192 -> 2048 -> 3648 columns, 1 row 16.0 / 13.8, 2 17.7 /
// 13.8, 8 17.9 / 15.3, 16 22.8 / 20.3; 2048 -> 2048 -> 2 x 8192 gated, 1 19.5 / 18.2, 8 21.7 / 19.4, 16 25.8 / 24.0; 14336 -> 4096 ->
// 6720, 1 36.2 / 36.3, 8 40.4 / 36.7, 16 45.8 / 42.6.  The norm in the second product's prologue instead, every workgroup norming the
// rows for itself (norm_gemv.hip), reads three times the bytes: as fast with 1 row, with 8 rows slower than the norm's own launch.
#include "sgemv_kernel.h"

using namespace k8sllm;

static bool rows_plan(int M, int N, int K, SmPlan& p) {
  return M >= 1 && M <= 16 && sm_min_m() <= 16 && sm_plan(M, N, K, false, false, p);
}

// floats of k-group partials; pair: W = [gate; up] of 2 N rows
extern "C" long long k8s_rows_workspace(int M, int N, int K, int pair) {
  SmPlan sp;
  if (N <= 0 || K <= 0 || !rows_plan(M, N, K, sp) || sp.g <= 1) return 0;
  return (long long)sp.g * M * N * (pair ? 2 : 1);
}

// y = x + mult a W^T, h = bf16(y (offset + nw)), sums [M][count] with room for 256 a row.  Returns count, or -5: a size or an alignment
// that this form does not take, nothing was launched.
extern "C" int k8s_rows_out(float* y, void* h, float* sums, const float* x, const void* nw, const void* a, const void* W, void* partial,
                            int M, int N, int K, float mult, float offset, hipStream_t stream) {
  if (!y || !h || !sums || !x || !nw || !a || !W || M < 1 || N <= 0 || K <= 0 || x == y) return -1;
  SmPlan sp;
  if (!rows_plan(M, N, K, sp) || ((uintptr_t)a | (uintptr_t)W) & 15 || (long long)M * K * 2 >= 1LL << 31) return -5;
  if (sp.g > 1 && partial == nullptr) return -3;
  SmRows r = {};
  r.x = x, r.y = y, r.h = (bf16_t*)h, r.nw = (const bf16_t*)nw, r.sums = sums, r.mult = mult, r.offset = offset;
  int count = 0;
  bool done = false;
#define RO(MT, JT)                                                                                                               \
  done = sm_launch<MT, JT, SG_F32, false, false, false, 1>(nullptr, partial, (const bf16_t*)a, W, nullptr, nullptr, M, N, K, 0.f, sp, \
                                                           stream, EpiAct{}, r, &count)
#define RO_JT(MT)              \
  if (sp.jt == 1) RO(MT, 1);      \
  else if (sp.jt == 2) RO(MT, 2); \
  else if (sp.jt == 4) RO(MT, 4); \
  else RO(MT, 8);
  if (M <= 8) { RO_JT(8) } else { RO_JT(16) }
#undef RO_JT
#undef RO
  if (!done) return -5;
  const int rc = (int)hipGetLastError();
  return rc != 0 ? -100 - rc : count;
}

// act(gain-less rms norm of the rows, times W^T) from h and sums as above.  kind: -1 (bf16; columns from n1 on go to out2), -2 (fp32) or
// a gated activation 0, 1, 5 of act.h (W [2 N][K]).
extern "C" int k8s_rows_in(void* out, void* out2, int n1, const void* h, const float* sums, int count, const void* W, void* partial,
                           int M, int N, int K, float eps, int kind, float limit, float alpha, hipStream_t stream) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (!out || !h || !sums || !W || M < 1 || N <= 0 || K <= 0 || (!pair && kind != -1 && kind != -2)) return -1;
  if (count < 1 || count > SM_SUMS || n1 <= 0 || n1 > N || (n1 < N && (out2 == nullptr || kind != -1))) return -1;
  SmPlan sp;
  if (!rows_plan(M, N, K, sp) || sp.jt > 4 || ((uintptr_t)h | (uintptr_t)W) & 15 || (long long)M * K * 2 >= 1LL << 31) return -5;
  if (sp.g > 1 && partial == nullptr) return -3;
  SmRows r = {};
  r.sums_in = sums, r.count = count, r.out2 = (bf16_t*)out2, r.n1 = n1;
  const EpiAct act{kind, limit, alpha};
  bool done = false;
#define RI(MT, JT, EE)                                                                                                          \
  done = sm_launch<MT, JT, EE, false, false, false, 2>(out, partial, (const bf16_t*)h, W, nullptr, nullptr, M, N, K, eps, sp, stream, \
                                                       act, r)
#define RI_JT(MT, EE)                 \
  if (sp.jt == 1) RI(MT, 1, EE);      \
  else if (sp.jt == 2) RI(MT, 2, EE); \
  else RI(MT, 4, EE);
#define RI_M(EE) \
  if (M <= 8) { RI_JT(8, EE) } else { RI_JT(16, EE) }
  if (pair) { RI_M(SG_GLU) } else if (kind == -2) { RI_M(SG_F32) } else { RI_M(SG_BF16) }
#undef RI_M
#undef RI_JT
#undef RI
  if (!done) return -5;
  return (int)hipGetLastError();
}

// out[g] = x[g] W_g^T for the first `groups` inputs x[g] [M][K], W_g of n rows, and out2 = tanh(x[groups] W_rest^T) of the rest rows of W
// [groups n + rest][K], bf16.  A launch of its own for the last one, which is small, cost it 6.7 us of a step.
extern "C" int k8s_rows_each(void* out, void* out2, const void* x, const void* W, int groups, int n, int rest, int M, int K,
                             hipStream_t stream) {
  if (!out || !out2 || !x || !W || groups < 1 || n < 1 || rest < 1 || M < 1 || K <= 0) return -1;
  SmPlan sp;
  if ((long long)groups * n + rest > 1 << 28 || !rows_plan(M, groups * n + rest, K, sp) || sp.jt > 4 || sp.g > 1 || n % 8 ||
      ((uintptr_t)x | (uintptr_t)W) & 15 || (long long)M * K * 2 >= 1LL << 31)
    return -5;
  const int N = groups * n + rest;
  SmRows r = {};
  r.out2 = (bf16_t*)out2, r.count = n, r.n1 = groups * n;
  bool done = false;
#define RE(MT, JT)                                                                                                                 \
  done = sm_launch<MT, JT, SG_BF16, false, false, false, 3>(out, nullptr, (const bf16_t*)x, W, nullptr, nullptr, M, N, K, 0.f, sp, stream, \
                                                            EpiAct{}, r)
#define RE_JT(MT)                 \
  if (sp.jt == 1) RE(MT, 1);      \
  else if (sp.jt == 2) RE(MT, 2); \
  else RE(MT, 4);
  if (M <= 8) { RE_JT(8) } else { RE_JT(16) }
#undef RE_JT
#undef RE
  if (!done) return -5;
  return (int)hipGetLastError();
}
