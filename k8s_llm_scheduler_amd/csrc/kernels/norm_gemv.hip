// One row times a weight matrix (bf16) with the norms ahead of it in the prologue: a decode step of a model with an fp32
// residual stream is a chain of small launches, and the norm between two products is one of them (3 - 4.5 us of the step, of
// which the work is a fraction).  Every workgroup normalises the row for itself -- 12 KB out of L2 at 2048 columns, while its
// first weights are on their way -- and workgroup 0 stores the new stream, to another buffer than the one the others still read.
//
//     y = x + mult b            or   y = x + b / rms(b) w1       (b: the last sublayer's output, bf16)
//     y = b / rms(b) w1 f(gate)                                   (no stream: b bf16 or fp32, f sigmoid or silu, optional)
//     h = y                     or   h = y / rms(y) (offset + nw) gain
//     out = act(bf16(h) W^T)                                      bf16, fp32 or an activation of act.h (gated: W = [gate; up])
//
// Bound by what the launch before it left in flight and by its own loads' way from memory.  us, two launches / one, weights from memory,
// inputs in the caches: 2048 -> 3648 7.9 / 6.3, 2048 (fp32 row with a gate) -> 2048 7.1 / 6.0, 2048 -> 8192 with an activation 10.2 /
// 8.9, 2048 -> 32768 fp32 24.7 / 23.1, 4096 -> 6720 14.1 / 12.9; a step of Katidra 447 -> 400.  Two rows are no gain (8.8 / 9.1, 11.1 /
// 12.7; the step 476 -> 480): every workgroup reads and norms both.
// Two rows of weights a wave from 4096 rows on (fewer waves, half the reads of the row from LDS), one below (more waves on a CU: the
// start is the longer part); at most 4 workgroups a CU, the waves of larger products take several sets of rows.
#include <type_traits>

#include "gemv_kernel.h"

namespace k8sllm {

struct NormGemvArgs {
  void* out;
  float* x_out;            // with x: the new stream [K]
  const float* x;          // [K] or null
  const void* branch;      // [K], bf16 or (b32) fp32
  const void* w1;          // of the branch's type, or null: no norm of it
  const bf16_t* gate;      // (no x) [K] or null
  const bf16_t* nw;        // or null: h = y
  const bf16_t* W;
  float mult, offset, gain, eps;
  int N_out, K, half_rows, per;   // per: row sets of a wave
  int b32, gate_silu;
  EpiAct act;
};

template <int RPW, int EPI>
__global__ void __launch_bounds__(256) norm_gemv_kernel(NormGemvArgs a) {
  constexpr int P = 2;                               // 8-element chunks of the row per thread (K <= 4096)
  constexpr int NR = gemv_paired(EPI) ? 2 * RPW : RPW, U = 4;
  __shared__ __attribute__((aligned(16))) u32x4 xs[P * 256];
  __shared__ float red[2][4];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int nch = a.K >> 3;

  // the row's loads, all of them ahead of the weights': loads retire in order
  f32x4 xa[P][2], bf[P][2], w1f[P][2];
  u32x4 bb[P], gg[P], w1b[P], nb[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = min(tid + 256 * p, nch - 1);
    if (a.x != nullptr) {
      const f32x4* r = reinterpret_cast<const f32x4*>(a.x) + 2 * c;
      xa[p][0] = r[0];
      xa[p][1] = r[1];
    }
    if (a.b32) {
      const f32x4* r = static_cast<const f32x4*>(a.branch) + 2 * c;
      bf[p][0] = r[0];
      bf[p][1] = r[1];
    } else {
      bb[p] = static_cast<const u32x4*>(a.branch)[c];
    }
    if (a.gate != nullptr) gg[p] = reinterpret_cast<const u32x4*>(a.gate)[c];
    if (a.w1 != nullptr) {
      if (a.b32) {
        const f32x4* r = static_cast<const f32x4*>(a.w1) + 2 * c;
        w1f[p][0] = r[0];
        w1f[p][1] = r[1];
      } else {
        w1b[p] = static_cast<const u32x4*>(a.w1)[c];
      }
    }
    if (a.nw != nullptr) nb[p] = reinterpret_cast<const u32x4*>(a.nw)[c];
  }
  // the first row set's weights
  const int sets = (a.N_out + RPW - 1) / RPW;
  int set = (int)blockIdx.x * 4 * a.per + wid;
  const int set_end = min(sets, ((int)blockIdx.x + 1) * 4 * a.per);
  auto row = [&](int s, int r) -> const u32x4* {     // weight row r of row set s (past the end: its last one)
    const int n = min(s * RPW + r % RPW, a.N_out - 1);
    return reinterpret_cast<const u32x4*>(a.W + (size_t)(r < RPW ? n : n + a.half_rows) * a.K);
  };
  u32x4 wv[U][NR];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int r = 0; r < NR; ++r) wv[u][r] = __builtin_nontemporal_load(row(set, r) + min(lane + 64 * u, nch - 1));
  asm volatile("" ::: "memory");

  auto bf_at = [](const u32x4& v, int e) { return e & 1 ? hi_bf(v[e >> 1]) : lo_bf(v[e >> 1]); };
  auto b_at = [&](int p, int e) { return a.b32 ? bf[p][e >> 2][e & 3] : bf_at(bb[p], e); };
  auto total = [&](float s, int slot) {              // over the workgroup (one barrier a slot)
    s = wave_sum(s);
    if (lane == 0) red[slot][wid] = s;
    __syncthreads();
    return red[slot][0] + red[slot][1] + red[slot][2] + red[slot][3];
  };
  float inv = a.mult;
  if (a.w1 != nullptr) {
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p)
      if (tid + 256 * p < nch) {
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(b_at(p, e), b_at(p, e), ss);
      }
    inv = 1.0f / sqrtf(total(ss, 0) / (float)a.K + a.eps);
  }
  float y[P][8], s2 = 0.f;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = tid + 256 * p;
    if (c >= nch) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float v = b_at(p, e) * inv;
      const float w = a.w1 == nullptr ? 1.f : a.b32 ? w1f[p][e >> 2][e & 3] : bf_at(w1b[p], e);
      if (a.x != nullptr) v = fmaf(v, w, xa[p][e >> 2][e & 3]);
      else v *= w;
      if (a.gate != nullptr) {
        const float g = bf_at(gg[p], e), s = 1.f / (1.f + expf(-g));
        v *= a.gate_silu ? g * s : s;
      }
      y[p][e] = v;
      s2 = fmaf(v, v, s2);
    }
    if (a.x_out != nullptr && blockIdx.x == 0) {
      f32x4* o = reinterpret_cast<f32x4*>(a.x_out) + 2 * c;
      o[0] = f32x4{y[p][0], y[p][1], y[p][2], y[p][3]};
      o[1] = f32x4{y[p][4], y[p][5], y[p][6], y[p][7]};
    }
  }
  float scale = 1.f;
  if (a.nw != nullptr) scale = a.gain / sqrtf(total(s2, 1) / (float)a.K + a.eps);
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = tid + 256 * p;
    if (c >= nch) continue;
    float h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = a.nw != nullptr ? y[p][e] * (scale * (a.offset + bf_at(nb[p], e))) : y[p][e];
    xs[c] = u32x4{pack_bf2(h[0], h[1]), pack_bf2(h[2], h[3]), pack_bf2(h[4], h[5]), pack_bf2(h[6], h[7])};
  }
  __syncthreads();

  // the weight stream: blocks of U chunks a lane, the next one (of this row set or the wave's next) under way while one is used
  float acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = 0.f;
  const int bpr = (nch + 64 * U - 1) / (64 * U);
  for (int j = 0; set < set_end;) {
    u32x4 cur[U][NR];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < NR; ++r) cur[u][r] = wv[u][r];
    int nj = j + 1, nset = set;
    if (nj == bpr) {
      nj = 0;
      nset = set + 4;
    }
    if (nset < set_end) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < NR; ++r)
          wv[u][r] = __builtin_nontemporal_load(row(nset, r) + min(nj * 64 * U + lane + 64 * u, nch - 1));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = j * 64 * U + lane + 64 * u;
      if (c < nch) {
        const u32x4 xv = xs[c];
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[r] = dot8(cur[u][r], xv, acc[r]);
      }
    }
    if (nj == 0) {                                   // row set `set` is complete
#pragma unroll
      for (int r = 0; r < NR; ++r) acc[r] = wave_sum(acc[r]);
      if (lane == 0) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
          const int n = set * RPW + r;
          if (n >= a.N_out) break;
          if constexpr (EPI == EPI_F32) static_cast<float*>(a.out)[n] = acc[r];
          else static_cast<bf16_t*>(a.out)[n] = f2bf(gemv_value<EPI>(acc[r], gemv_paired(EPI) ? acc[NR - RPW + r] : 0.f, a.act));
        }
      }
#pragma unroll
      for (int r = 0; r < NR; ++r) acc[r] = 0.f;
      set = nset;
    }
    j = nj;
  }
}

}  // namespace k8sllm

using namespace k8sllm;

// kind: -1 (bf16), -2 (fp32) or an activation: gated 0, 1, 5 (W [2 N_out][K]) or 7.  -5: a size or an alignment that this form does
// not take; nothing was launched.
extern "C" int k8s_norm_gemv(void* out, float* x_out, const float* x, const void* branch, int b32, const void* w1, float mult,
                             const void* gate, int gate_silu, const void* nw, float offset, float gain, float eps, const void* W,
                             int N_out, int K, int kind, float limit, float alpha, hipStream_t stream) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (out == nullptr || branch == nullptr || W == nullptr || N_out <= 0 || K <= 0 || (!pair && kind != 7 && kind != -1 && kind != -2))
    return -1;
  if ((x == nullptr) != (x_out == nullptr) || (x != nullptr && (x == x_out || b32 || gate != nullptr)) || (x == nullptr && w1 == nullptr))
    return -1;
  if (K % 8 || K > 4096 || N_out > (1 << 28)) return -5;
  if (((uintptr_t)x | (uintptr_t)x_out | (uintptr_t)branch | (uintptr_t)w1 | (uintptr_t)gate | (uintptr_t)nw | (uintptr_t)W) & 15) return -5;
  NormGemvArgs a = {out, x_out, x, branch, w1, (const bf16_t*)gate, (const bf16_t*)nw, (const bf16_t*)W, mult, offset, gain, eps,
                    N_out, K, pair ? N_out : 0, 1, b32, gate_silu, EpiAct{kind, limit, alpha}};
  auto go = [&](auto r, auto e) {
    constexpr int RR = decltype(r)::value, EE = decltype(e)::value;
    const int waves = (N_out + RR - 1) / RR, wgs = (waves + 3) / 4;
    a.per = (wgs + 1023) / 1024;
    norm_gemv_kernel<RR, EE><<<(wgs + a.per - 1) / a.per, 256, 0, stream>>>(a);
    return (int)hipGetLastError();
  };
  using std::integral_constant;
  auto by_rows = [&](auto e) {
    constexpr bool two = gemv_paired(decltype(e)::value);       // gate and up: two weight rows with one output of each
    if (!two && N_out >= 4096) return go(integral_constant<int, 2>{}, e);
    return go(integral_constant<int, 1>{}, e);
  };
  if (pair) return by_rows(integral_constant<int, EPI_GLU>{});
  if (kind == 7) return by_rows(integral_constant<int, EPI_ELEM>{});
  if (kind == -2) return by_rows(integral_constant<int, EPI_F32>{});
  return by_rows(integral_constant<int, EPI_BF16>{});
}
