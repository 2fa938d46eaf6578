// Windowed attention of prompt portions in true fp32 on the matrix cores (v_mfma_f32_16x16x4_f32: fp32 products and sums).
//
// The 16 columns of the products are 16 / R consecutive tokens of a sequence with the R query heads of one key head:
//   S^T[key][column] = K Q^T, O^T[dim][column] += V^T P^T, laid out as in latent_f32.hip: rows come from the cache as fragments, the
//   values pass through the wave's own LDS rows, the probabilities stay in the lanes that computed them.
// The 4 waves take the tiles of 16 keys in turn, without a barrier, and meet at the end; the next tile's rows are under way while the
// second product runs.  A value that one of the tokens does not see never meets its sums, be it an infinity or NaN: tiles at the edge of a
// token's keys run the second product token by token, with the values that it does not see as zeros.
// Bound by the fp32 matrix rate (a tile is 64 products of 32 cycles at 128 dimensions) and the loads' way where there are few tiles.
// us, plain FMAs (a workgroup a token, keys in LDS) / here, 16 heads over 4 of 128, window 1024: 300 tokens 144 / 28, 2 x 100 behind 400
// 221 / 29, 512 behind 500 861 / 73, 97 behind 1000 251 / 50, 24 fresh 17 / 11, 24 behind 1000 66 / 44; 32 over 8, 300 tokens 239 / 38.  Few
// tokens behind many keys, which a workgroup walks by itself, are left to that kernel's key splits (2 behind 3000 59 / 104) by
// ops/seqmix.py window_f32_plain.
#include "common.h"

namespace k8sllm {

template <int D>
__global__ __launch_bounds__(256, 2) void window_f32_kernel(
    float* __restrict__ out, const float* __restrict__ q, long ldq, const float* __restrict__ gate, long ldg,
    const float* __restrict__ kcache, const float* __restrict__ vcache, const int* __restrict__ block_tables, int max_blocks,
    const int* __restrict__ cu_q, const int* __restrict__ tok_seq, const int* __restrict__ positions, int T, int H, int G, int window, float scale, int sink, int bs, int chunk,
    float softcap, const float* __restrict__ sinkv, int gate_ph, const float* __restrict__ slopes) {
  constexpr int NS = D / 16, NT = D / 64, LD = D + 4;
  __shared__ __attribute__((aligned(16))) float rows[4][16][LD];       // a wave's tile of values; at the end its sums
  __shared__ float ml[4][16][2];
  const int R = H / G, NTK = 16 / R, kh = blockIdx.y, seq = blockIdx.z;
  const int tq0 = cu_q[seq] + blockIdx.x * NTK, end = cu_q[seq + 1], n = min(NTK, end - tq0);
  if (seq + 1 == (int)gridDim.z && blockIdx.x == 0)     // rows behind the last sequence: as idle ones
    for (int i = threadIdx.x; i < (T - end) * R * D; i += 256)
      out[((size_t)(end + i / (R * D)) * H + kh * R) * D + i % (R * D)] = 0.f;
  if (n <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, g = lane >> 4;
  const int pf = positions[tq0], pl = pf + n - 1;
  if (pf < 0) {                      // idle rows: defined output, nothing read
    for (int i = tid; i < n * R * D; i += 256) out[((size_t)(tq0 + i / (R * D)) * H + kh * R) * D + i % (R * D)] = 0.f;
    return;
  }
  const auto first = [&](int p) { return chunk > 0 ? p - p % chunk : window > 0 ? max(0, p - window + 1) : 0; };
  const int lo = first(pf), tiles = (pl - lo) / 16 + 1;              // first() does not fall with p
  const int tok = min(li / R, n - 1), hd = kh * R + li % R, p = pf + tok, lp = first(p);     // this lane's column (past the last: repeats)
  const int edge_lo = first(pl);     // keys from here to pf are seen by every token
  const int* btr = block_tables + (size_t)tok_seq[tq0] * max_blocks;
  const auto row_of = [&](int tile) {
    const int j = min(lo + tile * 16 + li, pl);
    return ((size_t)btr[j / bs] * bs + j % bs) * G * D + (size_t)kh * D + 4 * g;
  };
  f32x4 qf[NS], kf[NS], vf[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const f32x4*>(q + (size_t)(tq0 + tok) * ldq + (size_t)hd * D + 16 * s + 4 * g);
  const auto load = [&](size_t r) {
#pragma unroll
    for (int s = 0; s < NS; ++s) kf[s] = *reinterpret_cast<const f32x4*>(kcache + r + 16 * s);
#pragma unroll
    for (int s = 0; s < NS; ++s) vf[s] = *reinterpret_cast<const f32x4*>(vcache + r + 16 * s);
  };
  f32x4 o[NT][4];                    // o[x][e][i] = dimension 64 x + 16 g + 4 i + e of column li
#pragma unroll
  for (int x = 0; x < NT; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[x][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float slope = slopes != nullptr ? slopes[hd] : 0.f;
  float m = -INFINITY, l = 0.f;
  float(*mine)[LD] = rows[wave];
  if (wave < tiles) load(row_of(wave));
  for (int tile = wave; tile < tiles; tile += 4) {
    const int j0 = lo + tile * 16;
    f32x4 sc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) sc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s][e], qf[s][e], sc[e], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < NS; ++s) *reinterpret_cast<f32x4*>(&mine[li][16 * s + 4 * g]) = vf[s];
    asm volatile("" ::: "memory");                 // other lanes read what this one wrote
    if (tile + 4 < tiles) load(row_of(tile + 4));
    f32x4 w = (sc[0] + sc[1]) + (sc[2] + sc[3]);   // key j0 + 4 g + i, column li
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = j0 + 4 * g + i;
      float v = w[i] * scale;
      if (softcap > 0.f) v = softcap * tanhf(v / softcap);
      if (slopes != nullptr) v -= slope * (float)(p - j);
      w[i] = j >= lp && j <= p ? v : -INFINITY;
      top = fmaxf(top, w[i]);
    }
    top = lane_max<16>(top);
    top = lane_max<32>(top);
    const float mn = fmaxf(m, top), ref = mn == -INFINITY ? 0.f : mn;            // a column that has seen nothing yet
    const float alpha = m == -INFINITY ? 0.f : expf(m - ref);
    m = mn;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = expf(w[i] - ref);
      sum += w[i];
    }
    l = l * alpha + sum;
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int x = 0; x < NT; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[x][e] *= alpha;
    }
    if (j0 >= edge_lo && j0 + 15 <= pf) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int x = 0; x < NT; ++x) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(&mine[4 * g + s][64 * x + 4 * li]);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[x][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], w[s], o[x][e], 0, 0, 0);
        }
    } else {
      for (int k = 0; k < n; ++k) {
        const int pk = pf + k, lk = first(pk);
#pragma unroll
        for (int x = 0; x < NT; ++x) {
          f32x4 y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = o[x][e];
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const int j = j0 + 4 * g + s;
            f32x4 v = *reinterpret_cast<const f32x4*>(&mine[4 * g + s][64 * x + 4 * li]);
            if (j < lk || j > pk) v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], w[s], y[e], 0, 0, 0);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[x][e][i] = tok == k ? y[e][i] : o[x][e][i];
        }
      }
    }
  }
  l = lane_sum<16>(l);
  l = lane_sum<32>(l);
  if (g == 0) {
    ml[wave][li][0] = m;
    ml[wave][li][1] = l;
  }
  __syncthreads();
  const float s0 = !sink ? -INFINITY : sinkv != nullptr ? sinkv[hd] : 0.f;
  float M = s0;
#pragma unroll
  for (int x = 0; x < 4; ++x) M = fmaxf(M, ml[x][li][0]);
  const float part = m == -INFINITY ? 0.f : expf(m - M);           // a wave without keys: nothing
#pragma unroll
  for (int x = 0; x < NT; ++x)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4*>(&mine[li][64 * x + 16 * g + 4 * i]) = f32x4{o[x][0][i], o[x][1][i], o[x][2][i], o[x][3][i]} * part;
  __syncthreads();
  for (int i = tid; i < n * R * (D / 4); i += 256) {
    const int c = i / (D / 4), d = 4 * (i - c * (D / 4)), head = kh * R + c % R;
    const size_t t = tq0 + c / R;
    const float sk = !sink ? -INFINITY : sinkv != nullptr ? sinkv[head] : 0.f;
    float top = sk;
#pragma unroll
    for (int x = 0; x < 4; ++x) top = fmaxf(top, ml[x][c][0]);
    float den = sink ? expf(sk - top) : 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (ml[x][c][0] != -INFINITY) den += expf(ml[x][c][0] - top) * ml[x][c][1];
    f32x4 y = *reinterpret_cast<const f32x4*>(&rows[0][c][d]);
#pragma unroll
    for (int x = 1; x < 4; ++x) y += *reinterpret_cast<const f32x4*>(&rows[x][c][d]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = y[e] / den;
      if (gate != nullptr) v *= 1.f / (1.f + expf(-gate[t * ldg + (gate_ph ? (size_t)head : (size_t)head * D + d + e)]));
      y[e] = v;
    }
    *reinterpret_cast<f32x4*>(out + (t * H + head) * D + d) = y;
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" int k8s_window_f32_ok(int H, int G, int D, int V) {
  return G > 0 && H > 0 && H % G == 0 && 16 % (H / G) == 0 && D == V && (D == 64 || D == 128) && G <= 65535;
}

// cu_q: the query offsets of nseq sequences of at most max_qlen tokens at consecutive positions; tok_seq [T]: a token's row of the block
// tables (a sequence's first token's is read).
extern "C" int k8s_window_f32(float* out, const float* q, long ldq, const float* gate, long ldg, const float* kcache, const float* vcache,
                              const int* block_tables, int max_blocks, const int* cu_q, const int* tok_seq, const int* positions, int T,
                              int nseq, int max_qlen, int H, int G, int D, int V, int window, float scale, int sink, int bs, int chunk, float softcap,
                              const float* sinkv, int gate_ph, const float* slopes, hipStream_t s) {
  if (!k8s_window_f32_ok(H, G, D, V) || bs <= 0 || ldq % 4 || (((uintptr_t)out | (uintptr_t)q | (uintptr_t)kcache | (uintptr_t)vcache) & 15))
    return -1;
  if (nseq <= 0 || max_qlen <= 0) return 0;
  if (nseq > 65535) return -2;
  const int ntk = 16 / (H / G);
  const dim3 grid((max_qlen + ntk - 1) / ntk, G, nseq);
#define K8S_WF(DD)                                                                                                                \
  window_f32_kernel<DD><<<grid, 256, 0, s>>>(out, q, ldq, gate, ldg, kcache, vcache, block_tables, max_blocks, cu_q, tok_seq, \
                                             positions, T, H, G, \
                                             window, scale, sink, bs, chunk, softcap, sinkv, gate_ph, slopes)
  if (D == 64) K8S_WF(64);
  else K8S_WF(128);
#undef K8S_WF
  return (int)hipGetLastError();
}
