// One or two rows times a weight matrix (bf16) with the norms ahead of it in the prologue: a decode step of a model with an fp32
// residual stream is a chain of small launches, and the norm between two products is one of them (3 - 4.5 us of the step, of
// which the work is a fraction).  Every workgroup normalises the rows for itself -- M x 12 KB out of L2 at 2048 columns, while its
// first weights are on their way -- and workgroup 0 stores the new stream, to another buffer than the one the others still read.
//
//     y = x + mult b            or   y = x + b / rms(b) w1       (b: the last sublayer's output, bf16)
//     y = b / rms(b) w1 f(gate)                                   (no stream: b bf16 or fp32, f sigmoid or silu, optional)
//     h = y                     or   h = y / rms(y) (offset + nw) gain
//     out = act(bf16(h) W^T)                                      bf16, fp32 or an activation of act.h (gated: W = [gate; up])
//
// Bound by what the launch before it left in flight and by its own loads' way from memory: us, two launches / one (weights from
// memory, one row): 8192 x 2048 10.3 / 7.3, 2128 x 2048 8.6 / 5.2, 2048 x 2048 (fp32 rows with a gate) 8.9 / 5.3; 32768 x 2048 fp32 25.6 / 21.9.
// Two rows of weights a wave from 4096 rows on (fewer waves, half the reads of the rows from LDS), one below (more waves on a CU: the
// start is the longer part); at most 4 workgroups a CU, the waves of larger products take several sets of rows.
#include <type_traits>

#include "gemv_kernel.h"

namespace k8sllm {

struct NormGemvArgs {
  void* out;
  float* x_out;            // with x: the new stream [M][K]
  const float* x;          // [M][K] or null
  const void* branch;      // [M] rows of K, ldb elements apart; bf16, or (b32) fp32
  long ldb;
  const void* w1;          // of the branch's type, or null: no norm of it
  const bf16_t* gate;      // (no x) [M] rows of K, ldg apart, or null
  long ldg;
  const bf16_t* nw;        // or null: h = y
  const bf16_t* W;
  float mult, offset, gain, eps;
  int N_out, K, half_rows, per;   // per: row sets of a wave
  int b32, gate_silu;
  EpiAct act;
};

template <int M, int RPW, int EPI>
__global__ void __launch_bounds__(256) norm_gemv_kernel(NormGemvArgs a) {
  constexpr int P = 2;                               // 8-element chunks of a row per thread (K <= 4096)
  constexpr int NR = gemv_paired(EPI) ? 2 * RPW : RPW, U = 4;
  __shared__ __attribute__((aligned(16))) u32x4 xs[M][P * 256];
  __shared__ float red[2][4][M];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int nch = a.K >> 3;

  // the rows' loads, all of them ahead of the weights': loads retire in order
  f32x4 xa[P][M][2], bf[P][M][2];
  u32x4 bb[P][M], gg[P][M], w1b[P], nb[P];
  f32x4 w1f[P][2];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = min(tid + 256 * p, nch - 1);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (a.x != nullptr) {
        const f32x4* r = reinterpret_cast<const f32x4*>(a.x + (size_t)m * a.K) + 2 * c;
        xa[p][m][0] = r[0];
        xa[p][m][1] = r[1];
      }
      if (a.b32) {
        const f32x4* r = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.branch) + m * a.ldb) + 2 * c;
        bf[p][m][0] = r[0];
        bf[p][m][1] = r[1];
      } else {
        bb[p][m] = reinterpret_cast<const u32x4*>(static_cast<const bf16_t*>(a.branch) + m * a.ldb)[c];
      }
      if (a.gate != nullptr) gg[p][m] = reinterpret_cast<const u32x4*>(a.gate + m * a.ldg)[c];
    }
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

  auto b_of = [&](int p, int m, int e) -> float {
    return a.b32 ? bf[p][m][e >> 2][e & 3] : e & 1 ? hi_bf(bb[p][m][e >> 1]) : lo_bf(bb[p][m][e >> 1]);
  };
  // the rows' sums over the workgroup (slot: one barrier each)
  auto total = [&](float (&s)[M], int slot) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
      s[m] = wave_sum(s[m]);
      if (lane == 0) red[slot][wid][m] = s[m];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) s[m] = red[slot][0][m] + red[slot][1][m] + red[slot][2][m] + red[slot][3][m];
  };
  float inv[M];
#pragma unroll
  for (int m = 0; m < M; ++m) inv[m] = a.mult;
  if (a.w1 != nullptr) {
    float ss[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      ss[m] = 0.f;
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (tid + 256 * p < nch) {
#pragma unroll
          for (int e = 0; e < 8; ++e) ss[m] = fmaf(b_of(p, m, e), b_of(p, m, e), ss[m]);
        }
    }
    total(ss, 0);
#pragma unroll
    for (int m = 0; m < M; ++m) inv[m] = 1.0f / sqrtf(ss[m] / (float)a.K + a.eps);
  }
  float y[P][M][8], s2[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    s2[m] = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int c = tid + 256 * p;
      if (c >= nch) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = b_of(p, m, e) * inv[m];
        const float w = a.w1 == nullptr ? 1.f : a.b32 ? w1f[p][e >> 2][e & 3] : e & 1 ? hi_bf(w1b[p][e >> 1]) : lo_bf(w1b[p][e >> 1]);
        if (a.x != nullptr) v = fmaf(v, w, xa[p][m][e >> 2][e & 3]);
        else v *= w;
        if (a.gate != nullptr) {
          const float g = e & 1 ? hi_bf(gg[p][m][e >> 1]) : lo_bf(gg[p][m][e >> 1]);
          const float s = 1.f / (1.f + expf(-g));
          v *= a.gate_silu ? g * s : s;
        }
        y[p][m][e] = v;
        s2[m] = fmaf(v, v, s2[m]);
      }
      if (a.x_out != nullptr && blockIdx.x == 0) {
        f32x4* o = reinterpret_cast<f32x4*>(a.x_out + (size_t)m * a.K) + 2 * c;
        o[0] = f32x4{y[p][m][0], y[p][m][1], y[p][m][2], y[p][m][3]};
        o[1] = f32x4{y[p][m][4], y[p][m][5], y[p][m][6], y[p][m][7]};
      }
    }
  }
  if (a.nw != nullptr) total(s2, 1);
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const float s = a.nw != nullptr ? a.gain / sqrtf(s2[m] / (float)a.K + a.eps) : 1.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int c = tid + 256 * p;
      if (c >= nch) continue;
      float h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        h[e] = a.nw != nullptr ? y[p][m][e] * (s * (a.offset + (e & 1 ? hi_bf(nb[p][e >> 1]) : lo_bf(nb[p][e >> 1])))) : y[p][m][e];
      xs[m][c] = u32x4{pack_bf2(h[0], h[1]), pack_bf2(h[2], h[3]), pack_bf2(h[4], h[5]), pack_bf2(h[6], h[7])};
    }
  }
  __syncthreads();

  // the weight stream: blocks of U chunks a lane, the next one (of this row set or the wave's next) under way while one is used
  float acc[NR][M];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
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
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const u32x4 xv = xs[m][c];
#pragma unroll
          for (int r = 0; r < NR; ++r) acc[r][m] = dot8(cur[u][r], xv, acc[r][m]);
        }
      }
    }
    if (nj == 0) {                                   // row set `set` is complete
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = wave_sum(acc[r][m]);
      if (lane == 0) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
          const int n = set * RPW + r;
          if (n >= a.N_out) break;
#pragma unroll
          for (int m = 0; m < M; ++m) {
            if constexpr (EPI == EPI_F32) static_cast<float*>(a.out)[(size_t)m * a.N_out + n] = acc[r][m];
            else
              static_cast<bf16_t*>(a.out)[(size_t)m * a.N_out + n] =
                  f2bf(gemv_value<EPI>(acc[r][m], gemv_paired(EPI) ? acc[NR - RPW + r][m] : 0.f, a.act));
          }
        }
      }
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
      set = nset;
    }
    j = nj;
  }
}

}  // namespace k8sllm

using namespace k8sllm;

// kind: -1 (bf16), -2 (fp32) or an activation: gated 0, 1, 5 (W [2 N_out][K]) or 7.  -5: a size or an alignment that this form does
// not take; nothing was launched.
extern "C" int k8s_norm_gemv(void* out, float* x_out, const float* x, const void* branch, long ldb, int b32, const void* w1, float mult,
                             const void* gate, long ldg, int gate_silu, const void* nw, float offset, float gain, float eps,
                             const void* W, int M, int N_out, int K, int kind, float limit, float alpha, hipStream_t stream) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (out == nullptr || branch == nullptr || W == nullptr || M < 1 || N_out <= 0 || K <= 0 || (!pair && kind != 7 && kind != -1 && kind != -2))
    return -1;
  if ((x == nullptr) != (x_out == nullptr) || (x != nullptr && (x == x_out || b32 || gate != nullptr)) || (x == nullptr && w1 == nullptr))
    return -1;
  const int bb = b32 ? 4 : 2;
  if (M > 2 || K % 8 || K > 4096 || ldb * bb % 16 || (gate != nullptr && ldg % 8) || (M > 1 && ldb < K) || N_out > (1 << 28)) return -5;
  if (((uintptr_t)x | (uintptr_t)x_out | (uintptr_t)branch | (uintptr_t)w1 | (uintptr_t)gate | (uintptr_t)nw | (uintptr_t)W) & 15) return -5;
  NormGemvArgs a = {out, x_out, x, branch, ldb, w1, (const bf16_t*)gate, ldg, (const bf16_t*)nw, (const bf16_t*)W, mult, offset, gain, eps,
                    N_out, K, pair ? N_out : 0, 1, b32, gate_silu, EpiAct{kind, limit, alpha}};
  auto go = [&](auto m, auto r, auto e) {
    constexpr int MM = decltype(m)::value, RR = decltype(r)::value, EE = decltype(e)::value;
    const int waves = (N_out + RR - 1) / RR, wgs = (waves + 3) / 4;
    a.per = (wgs + 1023) / 1024;
    norm_gemv_kernel<MM, RR, EE><<<(wgs + a.per - 1) / a.per, 256, 0, stream>>>(a);
    return (int)hipGetLastError();
  };
  using std::integral_constant;
  auto by_rows = [&](auto m, auto e) {
    constexpr bool two = gemv_paired(decltype(e)::value);       // gate and up: two weight rows with one output of each
    if (!two && N_out >= 4096) return go(m, integral_constant<int, 2>{}, e);
    return go(m, integral_constant<int, 1>{}, e);
  };
  auto by_m = [&](auto e) { return M == 1 ? by_rows(integral_constant<int, 1>{}, e) : by_rows(integral_constant<int, 2>{}, e); };
  if (pair) return by_m(integral_constant<int, EPI_GLU>{});
  if (kind == 7) return by_m(integral_constant<int, EPI_ELEM>{});
  if (kind == -2) return by_m(integral_constant<int, EPI_F32>{});
  return by_m(integral_constant<int, EPI_BF16>{});
}
