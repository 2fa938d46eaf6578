// Latent attention over the paged cache in true fp32 on the matrix cores (v_mfma_f32_16x16x4_f32: fp32 products and sums).
//
// All heads of a token attend the same cached rows, so up to 16 of them are the columns of one product:
//   S^T[key][head] = K Q^T        A = 16 cached rows, loaded as the fragments they are; B = [q_abs | q_rot], in registers and LDS throughout
//   O^T[dim][head] += C^T P^T     A = the rows' latent dimensions, through the wave's own LDS rows; B = the probabilities as the
//                                 first product leaves them (step s of a tile takes the keys 4 g + s, so nothing crosses lanes)
// A workgroup is a token and 16 heads; its 4 waves take the tiles of 16 keys in turn, each with a maximum and sums of its own and no
// barrier, and meet at the end.  The next tile's rows are under way while the second product runs.  A wave holds queries, rows and
// sums of 512 + 64 dimensions in registers (one wave a SIMD), which is why a workgroup has no more tokens.
// Bound by the fp32 matrix rate: a tile is 272 products of 32 cycles a wave.  us, plain FMAs (a workgroup a token, a wave a head, keys in LDS)
// / here, 16 heads over 512 + 64, window 1024: 125 tokens behind 940 3305 / 112, 64 behind 600 2110 / 77, 1 behind 600 2097 / 75, 512 behind 1500 3786 /
// 238, 24 fresh 126 / 18; 32 heads, 125 behind 940 6582 / 122.
#include "common.h"

namespace k8sllm {

template <int C, int R>
__global__ __launch_bounds__(256, 1) void latent_f32_kernel(
    float* __restrict__ out, const float* __restrict__ q_abs, const float* __restrict__ q, const float* __restrict__ cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ tok_seq, const int* __restrict__ positions, int H,
    int Dn, int window, float scale, int bs, const float* __restrict__ sinks, const float* __restrict__ gate, long ldg) {
  constexpr int L = C + R, NS = L / 16, NC = C / 16, NT = C / 64, LD = C + 4;
  __shared__ __attribute__((aligned(16))) float rows[4][16][LD];       // a wave's tile of latent rows; at the end its sums
  __shared__ float ml[4][16][2];
  constexpr int QR = C >= 512 ? 14 : NS;           // fragments of the queries in registers; the others fit LDS beside the rows
  __shared__ f32x4 ql[NS - QR + 1][64];
  const int t = blockIdx.x, h0 = blockIdx.y * 16, heads = min(16, H - h0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, g = lane >> 4;
  const int p = positions[t];
  if (p < 0) {                       // idle row: defined output, nothing read
    for (int i = tid; i < heads * C; i += 256) out[((size_t)t * H + h0) * C + i] = 0.f;
    return;
  }
  const int lo = window > 0 ? max(0, p - window + 1) : 0, tiles = (p - lo) / 16 + 1;
  const int* btr = block_tables + (size_t)tok_seq[t] * max_blocks;
  const auto row_of = [&](int tile) {              // keys past the last repeat it
    const int j = min(lo + tile * 16 + li, p);
    return cache + ((size_t)btr[j / bs] * bs + j % bs) * L + 4 * g;
  };
  // fragment s: dimensions 16 s + 4 g .. + 3 of head h0 + li (heads past the last repeat it), of key li
  f32x4 qf[QR], kf[NS];
  {
    const int hd = min(h0 + li, H - 1);
    const float *qa = q_abs + ((size_t)t * H + hd) * C + 4 * g, *qr = q + ((size_t)t * H + hd) * (Dn + R) + Dn + 4 * g;
#pragma unroll
    for (int s = 0; s < QR; ++s) qf[s] = *reinterpret_cast<const f32x4*>(s < NC ? qa + 16 * s : qr + 16 * (s - NC));
    for (int s = QR + wave; s < NS; s += 4) ql[s - QR][lane] = *reinterpret_cast<const f32x4*>(s < NC ? qa + 16 * s : qr + 16 * (s - NC));
  }
  if constexpr (QR < NS) __syncthreads();
  const auto load = [&](const float* r) {
#pragma unroll
    for (int s = 0; s < NS; ++s) kf[s] = *reinterpret_cast<const f32x4*>(r + 16 * s);
  };
  f32x4 o[NT][4];                    // o[x][e][i] = dimension 64 x + 16 g + 4 i + e of head li
#pragma unroll
  for (int x = 0; x < NT; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[x][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  float(*mine)[LD] = rows[wave];
  if (wave < tiles) load(row_of(wave));
  for (int tile = wave; tile < tiles; tile += 4) {
    int at = lane;
    asm volatile("" : "+v"(at));                   // the queries in LDS are read a tile at a time, not kept in registers after all
    f32x4 sc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) sc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const f32x4 qs = s < QR ? qf[s < QR ? s : 0] : ql[s < QR ? 0 : s - QR][at];
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s][e], qs[e], sc[e], 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < NC; ++s) *reinterpret_cast<f32x4*>(&mine[li][16 * s + 4 * g]) = kf[s];
    asm volatile("" ::: "memory");                 // other lanes read what this one wrote
    if (tile + 4 < tiles) load(row_of(tile + 4));
    f32x4 w = (sc[0] + sc[1]) + (sc[2] + sc[3]);   // key 4 g + i, head li
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = lo + tile * 16 + 4 * g + i <= p ? w[i] * scale : -INFINITY;
      top = fmaxf(top, w[i]);
    }
    top = lane_max<16>(top);
    top = lane_max<32>(top);
    const float mn = fmaxf(m, top), ref = mn == -INFINITY ? 0.f : mn;            // scores of -infinity so far: they weigh nothing
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
    // the wave's own rows, and LDS serves a wave in order: no barrier
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int x = 0; x < NT; ++x) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(&mine[4 * g + s][64 * x + 4 * li]);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[x][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], w[s], o[x][e], 0, 0, 0);
      }
  }
  l = lane_sum<16>(l);
  l = lane_sum<32>(l);
  if (g == 0) {
    ml[wave][li][0] = m;
    ml[wave][li][1] = l;
  }
  __syncthreads();
  float M = sinks != nullptr ? sinks[min(h0 + li, H - 1)] : -INFINITY;
#pragma unroll
  for (int x = 0; x < 4; ++x) M = fmaxf(M, ml[x][li][0]);
  const float part = m == -INFINITY ? 0.f : expf(m - M);           // a wave without keys: nothing
#pragma unroll
  for (int x = 0; x < NT; ++x)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4*>(&mine[li][64 * x + 16 * g + 4 * i]) = f32x4{o[x][0][i], o[x][1][i], o[x][2][i], o[x][3][i]} * part;
  __syncthreads();
  for (int i = tid; i < heads * (C / 4); i += 256) {
    const int h = i / (C / 4), d = 4 * (i - h * (C / 4)), hd = h0 + h;
    float top = sinks != nullptr ? sinks[hd] : -INFINITY;
#pragma unroll
    for (int x = 0; x < 4; ++x) top = fmaxf(top, ml[x][h][0]);
    float den = sinks != nullptr ? expf(sinks[hd] - top) : 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (ml[x][h][0] != -INFINITY) den += expf(ml[x][h][0] - top) * ml[x][h][1];
    float f = 1.f / den;
    if (gate != nullptr) f *= 1.f / (1.f + expf(-gate[(size_t)t * ldg + hd]));
    f32x4 y = *reinterpret_cast<const f32x4*>(&rows[0][h][d]);
#pragma unroll
    for (int x = 1; x < 4; ++x) y += *reinterpret_cast<const f32x4*>(&rows[x][h][d]);
    *reinterpret_cast<f32x4*>(out + ((size_t)t * H + hd) * C + d) = y * f;
  }
}

}  // namespace k8sllm

using namespace k8sllm;

// -2: sizes or alignments that the kernel does not take.
extern "C" int k8s_latent_f32(float* out, const float* q_abs, const float* q, const float* cache, const int* block_tables, int max_blocks,
                              const int* tok_seq, const int* positions, int T, int C, int R, int H, int Dn, int window, float scale,
                              int bs, const float* sinks, const float* gate, long ldg, hipStream_t s) {
  if (Dn % 4 || (((uintptr_t)out | (uintptr_t)q_abs | (uintptr_t)q | (uintptr_t)cache) & 15) || (H + 15) / 16 > 65535) return -2;
  const dim3 grid(T, (H + 15) / 16);
#define K8S_LF(CC, RR)                                                                                                          \
  if (C == CC && R == RR) {                                                                                                     \
    latent_f32_kernel<CC, RR><<<grid, 256, 0, s>>>(out, q_abs, q, cache, block_tables, max_blocks, tok_seq, positions, H, Dn,   \
                                                   window, scale, bs, sinks, gate, ldg);                                        \
    return (int)hipGetLastError();                                                                                              \
  }
  K8S_LF(512, 64)
  K8S_LF(256, 64)
  K8S_LF(128, 64)
  K8S_LF(128, 32)
  K8S_LF(64, 32)
#undef K8S_LF
  return -2;
}
