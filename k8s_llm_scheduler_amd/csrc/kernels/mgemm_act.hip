// 17 - 128 rows times a weight matrix with an activation in the epilogue: mgemm.hip's kernel and plans, bf16 weights.
#include "mgemm_kernel.h"

namespace {
template <int EPI, int C = 0>
int mg_act(const MgArgs& a, int cfg, hipStream_t s) {
  if constexpr (C < kMgNumCfgs) {
    if (cfg == C) return mg_launch<C, EPI, false, false, false>(a, a.nwg, s);
    return mg_act<EPI, C + 1>(a, cfg, s);
  } else {
    return -4;
  }
}
}  // namespace

// kind: gated 0, 1, 5 (W [2 N_out][K] = gate | up) or 7; the plan (cfg, nwg, cmax, slabs, tickets) as k8s_mgemm takes it with epi 2
// (gated) or 0.
extern "C" int k8s_mgemm_act(void* out, float* ws, unsigned* tickets, const void* x, const void* W, int M, int N_out, int K,
                             int cfg, int nwg, int cmax, int kind, float limit, float alpha, int fenced, hipStream_t stream) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (cfg < 0 || cfg >= kMgNumCfgs || M <= 0 || N_out <= 0 || N_out % 4 || K <= 0 || nwg <= 0 || cmax < 1) return -1;
  if (!pair && kind != 7) return -1;
  const long long kbytes = (long long)K * 2, wrows = pair ? 2LL * N_out : N_out;
  if (kbytes % kMgCfgs[cfg].rb != 0) return -1;
  const int epi = pair ? MG_SWIGLU : MG_BF16;
  const MgGeom g = mg_geom(M, N_out, K, epi, 0, cfg);
  if (nwg > g.total) return -1;
  if (cmax > 1 && (ws == nullptr || tickets == nullptr)) return -3;
  if (wrows * kbytes >= (1LL << 32) || (long long)M * kbytes >= (1LL << 32)) return -5;   // 32-bit DMA offsets
  MgArgs a = {};
  a.act = EpiAct{kind, limit, alpha};
  a.fenced = fenced;
  a.out = out;
  a.ws = ws;
  a.cnt = tickets;
  a.x = static_cast<const uint8_t*>(x);
  a.W = static_cast<const uint8_t*>(W);
  a.kbytes = a.xkbytes = kbytes;
  a.total = g.total;
  a.M = M;
  a.N_out = N_out;
  a.half_rows = pair ? N_out : 0;
  a.m_tiles = (M + kMgCfgs[cfg].bm - 1) / kMgCfgs[cfg].bm;
  a.T = (int)g.T;
  a.nwg = nwg;
  a.cmax = cmax;
  return pair ? mg_act<MG_GLU>(a, cfg, stream) : mg_act<MG_ELEM>(a, cfg, stream);
}
