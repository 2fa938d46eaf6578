// K3 / K8 / K9(+K10) / K11 / K15: hand-written MFMA GEMM for projections with more than 2 rows
// (prefill chunks, batched decode), bf16 or OCP-e4m3 weights, fp32 accumulate (gfx950).
//
//     out[M, N] = epi( x[M, K] . W[N, K]^T )        epi: bf16 | fp32 | SwiGLU (silu(g) * u)
//
// Design (MI355X-first, not a library tile recompiled):
//  * swapped orientation C^T = W . x^T on v_mfma_f32_16x16x32_bf16 (fp8: _16x16x32_fp8_fp8): the
//    A operand is 16 weight rows, the B operand 16 activation rows, both K-contiguous, so both are
//    staged the same way and every lane ends with 4 CONSECUTIVE output columns of one row
//    (one 8-byte bf16 / 16-byte fp32 store, and gate/up pairs side by side for SwiGLU).
//  * both operands move HBM/L2 -> LDS by LDS-DMA (global_load_lds_dwordx4): no VGPR staging, an
//    S-deep ring of 128-byte-wide k-steps (64 bf16 or 128 e4m3 per row), counted `s_waitcnt
//    vmcnt` so S-2 k-steps stay in flight across each raw s_barrier (MI355X_MICROARCH: LDS-DMA
//    stays in flight across barriers; __syncthreads would drain it).
//  * the LDS image is lane-linear (DMA destination = base + 16 * lane); the XOR swizzle that makes
//    the fragment reads (16 rows x one 16-byte column, ds_read_b128) conflict-free is applied on the
//    per-lane GLOBAL source address: 16-byte chunk c of row r lives at slot c ^ ((r >> 1) & 7).
//  * block -> tile mapping is XCD-aware (blocks b, b+8, .. share an XCD and get a contiguous
//    logical range), with the k-slices of one tile adjacent, then the m-tiles of one n-tile:
//    the weights a tile streams are re-read by its neighbours from the same L2.
//  * split-K for small grids (TP = 8 shapes: N = 1280, K = 8192): every slice writes an fp32 slab
//    in fragment order with write-through (sc1) 16-byte buffer stores, waits for them, and counts its
//    arrival with one relaxed device-scope ticket add; the last arriving slice of a tile reads all
//    slabs back with sc1 loads (fixed order), reduces them and applies the epilogue in the same launch
//    (no memset, no second kernel, no cache-wide fence; the ticket is reset by the reducer).  Measured
//    against the round-4 form (plain stores + agent-scope release / acquire fences, K8S_MGEMM_FENCED=1):
//    batch-64 decode 30.68 -> 30.46 ms/step bf16, 18.73 -> 18.30 fp8 (profiles/mgemm_fence_ab_r5.txt).
//  * fp8: activations are quantized per token (fp8.hip), weights per row; the epilogue applies
//    sx[m] * sw[n].  Non-scaled fp8 MFMA runs at the bf16 rate but halves the staged bytes.
//  * MX activations (host mode fp8 = 3): x is OCP MX e4m3 -- one E8M0 scale per 32 values of a row (fp8.hip), as
//    the SwiGLU epilogue below and the attention kernels write it -- and the MFMA is the block-scaled
//    v_mfma_scale_f32_16x16x128_f8f6f4: lane (li, g) holds k 16 g.. and 64 + 16 g.. of its row and passes the scale
//    byte of block g as its B scale (the weights' per-row scale stays in the epilogue, unit A scales).  The
//    scale bytes ride the x ring: one 4-byte LDS-DMA per (row, 128-value subtile) per k-step.  Twice the MFMA rate
//    of the non-scaled fp8 form, and no per-token absmax pass anywhere.
//  * MX output (SwiGLU epilogue, mx_out): the h = silu(g) * u values of 32 consecutive features of a row sit in
//    the lanes of one 16-lane column group of two adjacent fragments (the configurations whose per-wave feature
//    span is a multiple of 32), or of one fragment in each of two neighbouring waves (16 features per wave: the
//    row absmax goes through LDS, one barrier): a shuffle max gives the block's E8M0 scale and every lane stores
//    its e4m3 bytes -- the down projection's input is produced already quantized.
#include "mgemm_kernel.h"

namespace {
template <int C, bool FP8, bool MX>
int mg_epi(const MgArgs& a, int grid, int epi, bool mxo, hipStream_t s) {
  if constexpr (FP8) {   // MX output: the SwiGLU / residual epilogues of the fp8 and MX modes
    if (mxo) {
      if (epi == MG_SWIGLU) return mg_launch<C, MG_SWIGLU, FP8, MX, true>(a, grid, s);
      if (epi == MG_BF16) return mg_launch<C, MG_BF16, FP8, MX, true>(a, grid, s);
      return -2;
    }
  }
  switch (epi) {
    case MG_BF16: return mg_launch<C, MG_BF16, FP8, MX, false>(a, grid, s);
    case MG_F32: return mg_launch<C, MG_F32, FP8, MX, false>(a, grid, s);
    case MG_SWIGLU: return mg_launch<C, MG_SWIGLU, FP8, MX, false>(a, grid, s);
  }
  return -2;
}

template <bool FP8, bool MX, int C = 0>
int mg_cfg(const MgArgs& a, int grid, int cfg, int epi, bool mxo, hipStream_t s) {
  if constexpr (C < kMgNumCfgs) {
    if (cfg == C) return mg_epi<C, FP8, MX>(a, grid, epi, mxo, s);
    return mg_cfg<FP8, MX, C + 1>(a, grid, cfg, epi, mxo, s);
  } else {
    return -4;
  }
}

}  // namespace

extern "C" int k8s_mgemm_num_configs() { return kMgNumCfgs; }

namespace {
constexpr bool mg_mx_ok(int c) { return c < kMgNumCfgs && mg_mx_cfg(c); }
template <int C = 0>
bool mg_mx_valid(int cfg) {
  if constexpr (C < kMgNumCfgs) return cfg == C ? mg_mx_ok(C) : mg_mx_valid<C + 1>(cfg);
  else return false;
}
template <int C = 0>
bool mg_mxo_valid(int cfg) {
  if constexpr (C < kMgNumCfgs) return cfg == C ? mg_mxo_cfg(C) : mg_mxo_valid<C + 1>(cfg);
  else return false;
}
bool mg_mxr_valid(int cfg) { return cfg >= 0 && cfg < kMgNumCfgs && (kMgCfgs[cfg].bn / (kMgCfgs[cfg].wn * 16)) % 2 == 0; }
}  // namespace

// LDS bytes of a config in a mode (0 bf16, 1 fp8, 3 MX activations; 2 is not a mode); -1: the config is not built for
// that mode.  Mode 4: 0 if the config's SwiGLU epilogue can write MX output, else -1; mode 5: the same for the residual
// epilogue.
extern "C" int k8s_mgemm_lds_bytes(int cfg, int mode) {
  if (cfg < 0 || cfg >= kMgNumCfgs || mode < 0 || mode > 5 || mode == 2) return -1;
  if (mode == 4) return mg_mxo_valid(cfg) ? 0 : -1;
  if (mode == 5) return mg_mxr_valid(cfg) ? 0 : -1;
  const int b = mg_lds_bytes(kMgCfgs[cfg], mode);
  if (mode == 3 && !mg_mx_valid(cfg)) return -1;
  return b;
}

// (bm, bn) of a config: the Python planner sizes grids from them.
extern "C" int k8s_mgemm_config(int cfg, int* bm, int* bn, int* threads, int* lds_bytes, int* swiglu, int* rb) {
  if (cfg < 0 || cfg >= kMgNumCfgs) return -1;
  const MgCfg c = kMgCfgs[cfg];
  *bm = c.bm;
  *bn = c.bn;
  *threads = 64 * c.wm * c.wn * c.wk;
  *lds_bytes = c.s * (c.bm + c.bn) * c.rb + 16 + c.wk * c.wn * c.bm * 4;
  *swiglu = (c.bn / (c.wn * 16)) % 2 == 0;
  *rb = c.rb;
  return 0;
}

// Plan facts for a launch of `nwg` workgroups: the tile count, the most workgroups sharing one tile
// (cmax), the fp32 slab workspace (elements) and the ticket count.  Returns -1 for bad arguments.
extern "C" int k8s_mgemm_plan_info(int M, int N_out, int K, int epi, int fp8, int cfg, int nwg, long long* tiles,
                                   int* cmax, long long* ws_elems) {
  if (cfg < 0 || cfg >= kMgNumCfgs || M <= 0 || N_out <= 0 || K <= 0 || nwg <= 0) return -1;
  const MgGeom g = mg_geom(M, N_out, K, epi, fp8, cfg);
  if (g.T <= 0 || (long long)K * (fp8 ? 1 : 2) % kMgCfgs[cfg].rb != 0 || nwg > g.total) return -1;
  int cm = 1;
  for (long long t = 0; t < g.tiles; ++t) {
    const long long f = ((t * g.T + 1) * nwg - 1) / g.total, l = (((t + 1) * g.T) * nwg - 1) / g.total;
    if (l - f + 1 > cm) cm = (int)(l - f + 1);
  }
  *tiles = g.tiles;
  *cmax = cm;
  *ws_elems = cm > 1 ? g.tiles * cm * (kMgCfgs[cfg].bm * kMgCfgs[cfg].bn + kMgCfgs[cfg].bm) : 0;
  return 0;
}

// out[M, N_out] = epi(x[M, K] . W^T) with `nwg` workgroups streaming equal shares of the
// (tile, k-step) items.  fp8 = 1: x / W are e4m3 bytes with per-row scales xs / wsc; fp8 = 3 (MX): W e4m3 with row
// scales wsc, x MX e4m3 with its E8M0 block scales in xs (bytes, mx_scale_off layout).  oq / oe (fp8 = 1 or 3, SwiGLU): the
// output is written as MX e4m3 [M][N_out] + E8M0 (mx_scale_off layout) instead of bf16 (out unused).
// SwiGLU: W holds 2 * N_out rows ([gate; up]); out has N_out columns.
extern "C" int k8s_mgemm(void* out, float* ws, unsigned* tickets, const void* x, const void* W, const float* xs,
                         const float* wsc, int M, int N_out, int K, int epi, int fp8, int cfg, int nwg, int cmax,
                         const void* res, int rms, float eps, void* oq, void* oe, int fenced, hipStream_t stream) {
  if (cfg < 0 || cfg >= kMgNumCfgs || M <= 0 || N_out <= 0 || K <= 0 || nwg <= 0 || cmax < 1) return -1;
  if (N_out % 4 != 0) return -1;
  if (fp8 < 0 || fp8 > 3 || fp8 == 2) return -1;
  const bool mx = fp8 == 3, mxo = oq != nullptr;
  if (mxo && (oe == nullptr || (fp8 != 1 && fp8 != 3) || N_out % 128 != 0 ||
              !(epi == MG_SWIGLU ? mg_mxo_valid(cfg) : (epi == MG_BF16 && res != nullptr && mg_mxr_valid(cfg)))))
    return -7;
  if (mx && (K % 128 != 0 || !mg_mx_valid(cfg))) return -7;
  const long long kbytes = (long long)K * (fp8 ? 1 : 2), xkbytes = kbytes;
  if (kbytes % kMgCfgs[cfg].rb != 0) return -1;
  const MgGeom g = mg_geom(M, N_out, K, epi, fp8, cfg);
  if (nwg > g.total) return -1;
  if (cmax > 1 && (ws == nullptr || tickets == nullptr)) return -3;
  const long long wrows = epi == MG_SWIGLU ? 2LL * N_out : (long long)N_out;
  if (wrows * kbytes >= (1LL << 32) || (long long)M * xkbytes >= (1LL << 32)) return -5;  // 32-bit DMA offsets
  if ((fp8 == 1 || fp8 == 3) && (xs == nullptr || wsc == nullptr)) return -3;
  if (res != nullptr && epi != MG_BF16) return -6;   // residual epilogue: bf16 output only
  if (rms && fp8 == 1) return -6;   // per-token e4m3 activations carry 1 / rms in their scales (MX rows: prologue)
  MgArgs a;
  a.res = static_cast<const bf16_t*>(res);
  a.rms = rms;
  a.eps = eps;
  // RMS prologue on the MFMA for the wide projections (>= 8192 output features: the 70B TP = 1 / 2 QKV, gate/up),
  // v_dot2 squares for the narrow ones, where the extra MFMA is as large as the tile's own work (one TP = 8 rank:
  // batch-64 decode 7.66 ms/step with v_dot2, 7.78 with the MFMA; TP = 1: 31.98 -> 30.72, profiles/rms_mfma_ab_r5.txt).
  // K8S_RMS_MFMA = 0 / 1 forces one form.
  static const int rms_mfma_env = [] { const char* e = getenv("K8S_RMS_MFMA"); return e ? atoi(e) : -1; }();
  a.rms_mfma = rms_mfma_env >= 0 ? rms_mfma_env : (N_out >= 8192 ? 1 : 0);
  a.fenced = fenced;   // (ops.mgemm: K8S_MGEMM_FENCED, or per call in the fenced-vs-fence-free test)
  a.out = out;
  a.ws = ws;
  a.cnt = tickets;
  a.x = static_cast<const uint8_t*>(x);
  a.W = static_cast<const uint8_t*>(W);
  a.xs = xs;
  a.wsc = wsc;
  a.xe = mx ? reinterpret_cast<const uint8_t*>(xs) : nullptr;
  a.oq = static_cast<uint8_t*>(oq);
  a.oe = static_cast<uint8_t*>(oe);
  a.kbytes = kbytes;
  a.xkbytes = xkbytes;
  a.total = g.total;
  a.M = M;
  a.N_out = N_out;
  a.half_rows = epi == MG_SWIGLU ? N_out : 0;
  a.m_tiles = (M + kMgCfgs[cfg].bm - 1) / kMgCfgs[cfg].bm;
  a.T = (int)g.T;
  a.nwg = nwg;
  a.cmax = cmax;
  if (mx) return mg_cfg<true, true>(a, nwg, cfg, epi, mxo, stream);
  return fp8 ? mg_cfg<true, false>(a, nwg, cfg, epi, mxo, stream) : mg_cfg<false, false>(a, nwg, cfg, epi, false, stream);
}
