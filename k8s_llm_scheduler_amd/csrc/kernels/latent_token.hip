// Latent attention of single tokens (decoding): every token is another sequence, its queries absorbed into the latent space,
// the cached rows [normed latent (C) | rotated key part (R)] attended as they are stored.
#include "common.h"

namespace k8sllm {

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// Workgroups (token, group of 16 heads, key split) of 4 waves, 64 keys per step.  All rows of a step are in flight at once
// (18 vectors per thread, each thread's two page numbers ahead of them), staged in LDS, and the waves share the step both
// ways: the scores by keys, S^T = K Q^T for 16 keys each, and the value product by latent columns, O += P C for C / 4 columns
// each, the weights (bf16 for the product, summed in fp32) passing through LDS.  Every split leaves its maximum, sum and
// unnormalised O; latent_out_kernel joins them.  Bound by the latency of table, rows, LDS and products in turn: contexts of
// 529 tokens, 16 heads: 1 row 7.3 us, 8 rows 7.6 us (one wave per 32 keys with a row's address and load waited for in turn:
// 21 and 22 us).
template <int C, int R>
__global__ __launch_bounds__(256) void latent_token_kernel(
    float* __restrict__ pacc, float* __restrict__ pml, const bf16_t* __restrict__ q_abs, const bf16_t* __restrict__ q,
    const bf16_t* __restrict__ cache, const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ tok_seq,
    const int* __restrict__ positions, int H, int Dn, int window, float scale, int bs, int nsplit) {
  constexpr int L = C + R, NKK = L / 32, ROW = (L + 8) * 2, CPR = L / 8, NLD = CPR / 8, NB = C / 64, KT = 64;
  static_assert(L % 64 == 0 && C % 64 == 0, "whole pieces");
  extern __shared__ __attribute__((aligned(16))) char smem_t[];
  char* kl = smem_t;                                             // [64][L + 8] bf16
  bf16_t* pw = reinterpret_cast<bf16_t*>(smem_t + KT * ROW);     // weights [16 heads][64 + 8 keys]
  float* wm = reinterpret_cast<float*>(pw + 16 * (KT + 8));      // the waves' maxima, then sums: [4][16]
  const int t = blockIdx.x, hg = blockIdx.y, split = blockIdx.z, HP = gridDim.y * 16;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int p = positions[t], seq = tok_seq[t], lo = window > 0 ? max(0, p - window + 1) : 0;
  const int nsteps = p < 0 ? 0 : (p - lo + KT) / KT, per = (nsteps + nsplit - 1) / nsplit;
  const int s0 = split * per, s1 = min(nsteps, s0 + per);
  const size_t rec0 = ((size_t)t * HP + hg * 16) * nsplit + split;    // the head's record: rec0 + head * nsplit
  if (s0 >= s1) {                                                // nothing to see: no weight in the merge
    if (tid < 16) {
      pml[(rec0 + (size_t)tid * nsplit) * 2] = -INFINITY;
      pml[(rec0 + (size_t)tid * nsplit) * 2 + 1] = 0.f;
    }
    return;
  }
  const int* btr = block_tables + (size_t)seq * max_blocks;
  const int lr = tid >> 3, lc = tid & 7;                         // loader: rows lr, lr + 32, pieces lc + 8 i
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  u32x4 pre[2][NLD];
  auto fetch = [&](int step) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int key = min(lo + step * KT + lr + 32 * r, p);      // rows past the last key repeat it; their weights are zero
      const bf16_t* row = cache + ((size_t)btr[key / bs] * bs + key % bs) * L + 8 * lc;
#pragma unroll
      for (int i = 0; i < NLD; ++i) pre[r][i] = *reinterpret_cast<const u32x4*>(row + 64 * i);
    }
  };
  fetch(s0);
  bf16x8 qf[NKK];              // B operand of S^T = K Q^T: lane (li = head, g) holds [q_abs | q_rot][32 kk + 8 g .. + 7]
  {
    const int hd = hg * 16 + li;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      const int piece = 32 * kk + 8 * g;
      u32x4 v = zero;
      if (hd < H)
        v = piece < C ? *reinterpret_cast<const u32x4*>(q_abs + ((size_t)t * H + hd) * C + piece)
                      : *reinterpret_cast<const u32x4*>(q + ((size_t)t * H + hd) * (Dn + R) + Dn + (piece - C));
      qf[kk] = __builtin_bit_cast(bf16x8, v);
    }
  }
  f32x4 o[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;                          // head li; l_run: this wave's keys
  const int qd = li >> 2, pd = li & 3;
  for (int step = s0; step < s1; ++step) {
    if (step > s0) __syncthreads();                              // the last step's rows and weights have been read
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int i = 0; i < NLD; ++i) *reinterpret_cast<u32x4*>(kl + (lr + 32 * r) * ROW + 16 * (lc + 8 * i)) = pre[r][i];
    lds_barrier();
    if (step + 1 < s1) fetch(step + 1);
    const int j0 = lo + step * KT + 16 * wave + 4 * g;           // this lane's keys j0 .. j0 + 3
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      const bf16x8 ka = *reinterpret_cast<const bf16x8*>(kl + (16 * wave + li) * ROW + 64 * kk + 16 * g);
      s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[kk], s, 0, 0, 0);
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = j0 + i <= p ? s[i] * scale : -INFINITY;
      tmax = fmaxf(tmax, s[i]);
    }
    tmax = lane_max<16>(tmax);
    tmax = lane_max<32>(tmax);
    if (g == 0) wm[16 * wave + li] = tmax;
    lds_barrier();
    const float m_new = fmaxf(fmaxf(fmaxf(wm[li], wm[16 + li]), fmaxf(wm[32 + li], wm[48 + li])), m_run);   // finite
    const float alpha = m_run == -INFINITY ? 0.f : __expf(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
    bf16x4 pb;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float e = __expf(s[i] - m_new);
      l_run += e;
      pb[i] = (__bf16)e;
    }
    *reinterpret_cast<bf16x4*>(pw + li * (KT + 8) + 16 * wave + 4 * g) = pb;
    lds_barrier();
    if (step > s0) {
      float a_i[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a_i[i] = __shfl(alpha, 4 * g + i, WAVE);
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[n][i] *= a_i[i];
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const bf16x4 p0 = *reinterpret_cast<const bf16x4*>(pw + li * (KT + 8) + 32 * kb + 4 * g);
      const bf16x4 p1 = *reinterpret_cast<const bf16x4*>(pw + li * (KT + 8) + 32 * kb + 16 + 4 * g);
      bf16x8 pa;       // slot j < 4: key 4 g + j; slot j >= 4: key 16 + 4 g + (j - 4)
#pragma unroll
      for (int j = 0; j < 4; ++j) { pa[j] = p0[j]; pa[4 + j] = p1[j]; }
      const char* v0r = kl + (32 * kb + 4 * g + qd) * ROW;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const int col = (C / 4) * wave + 16 * n + 4 * pd;
        const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(v0r + 2 * col));
        const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(v0r + 16 * ROW + 2 * col));
        bf16x8 vb;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vb[j] = v0[j]; vb[4 + j] = v1[j]; }
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, vb, o[n], 0, 0, 0);
      }
    }
  }
  // o[n][i] = O[head 4 g + i][column C / 4 wave + 16 n + li]
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      pacc[(rec0 + (size_t)(4 * g + i) * nsplit) * C + (C / 4) * wave + 16 * n + li] = o[n][i];
  l_run = lane_sum<16>(l_run);
  l_run = lane_sum<32>(l_run);
  __syncthreads();
  if (g == 0) wm[16 * wave + li] = l_run;
  __syncthreads();
  if (tid < 16) {
    pml[(rec0 + (size_t)tid * nsplit) * 2] = m_run;
    pml[(rec0 + (size_t)tid * nsplit) * 2 + 1] = wm[tid] + wm[16 + tid] + wm[32 + tid] + wm[48 + tid];
  }
}

// The splits of up to 4 tokens joined and taken through the head's value up-projection in one launch: workgroups (head, 4
// tokens) of V / 16 waves.  lat[c] = sum_s e^(m_s - M) O_s[c] / sum_s e^(m_s - M) l_s (with a sink: one more term e^sink),
// times the head's gate, rounded to bf16 as the product's operand; out = lat W_uv^T with the tokens as the columns of the
// instruction's tile and the weights, loaded ahead of the merge, straight from memory as its rows.  nsplit <= 32.
// 16 splits, 16 heads: 4.8 us at 1 and 8 rows in quarters of the value columns, 7.3 with all of a head's.
// CB: blocks of 16 value columns of a workgroup, its waves sharing k where they are fewer than waves.
template <int C, int V, int CB>
__global__ __launch_bounds__(4 * V) void latent_out_kernel(bf16_t* __restrict__ out, const float* __restrict__ pacc,
                                                           const float* __restrict__ pml, const bf16_t* __restrict__ uv,
                                                           int T, int H, int HP, int nsplit,
                                                           const float* __restrict__ sinks,
                                                           const bf16_t* __restrict__ gate, long ldg) {
  constexpr int KS = V / 16 / CB, NKK = C / 32 / KS;   // shares of k, steps of a share
  static_assert(V == 128 && C == 512, "a thread per 4 latent columns and token");
  __shared__ float ws[4][32];
  __shared__ __attribute__((aligned(16))) bf16_t lat[16][C + 8];
  __shared__ __attribute__((aligned(16))) float part[KS > 1 ? KS : 1][CB][KS > 1 ? 64 : 1][4];
  const int hd = blockIdx.x % H, v0 = blockIdx.x / H * (16 * CB), t0 = blockIdx.y * 4, nt = min(4, T - t0);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int cb = wave % CB, kk0 = wave / CB * NKK;
  // everything is requested at once, in the order of its use (loads retire in order): maxima and sums, the first splits' sums, weights
  const int tw = t0 + min(wave, nt - 1);               // a wave per token, a lane per split
  const size_t rec = ((size_t)tw * HP + hd) * nsplit + min(lane, nsplit - 1);
  const float m0 = pml[2 * rec], l0 = pml[2 * rec + 1];
  const float g0 = gate != nullptr ? bf2f(gate[(size_t)tw * ldg + hd]) : 0.f;
  constexpr int AHEAD = 16;
  const int k = tid >> 7, c = 4 * (tid & 127);
  const float* pr = pacc + ((size_t)(t0 + min(k, nt - 1)) * HP + hd) * nsplit * C + c;
  f32x4 x[AHEAD];
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) x[u] = *reinterpret_cast<const f32x4*>(pr + (size_t)min(u, nsplit - 1) * C);
  bf16x8 wf[NKK];
  const bf16_t* wr = uv + ((size_t)hd * V + v0 + 16 * cb + li) * C + 32 * kk0 + 8 * g;
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) wf[kk] = *reinterpret_cast<const bf16x8*>(wr + 32 * kk);
  asm volatile("" ::: "memory");
  if (wave < nt) {
    const float m = lane < nsplit ? m0 : -INFINITY, l = lane < nsplit ? l0 : 0.f;
    float M = wave_max(m);
    if (sinks != nullptr) M = fmaxf(M, sinks[hd]);
    const float e = m == -INFINITY ? 0.f : expf(m - M);
    float den = wave_sum(e * l);
    if (sinks != nullptr) den += expf(sinks[hd] - M);
    const float gh = gate != nullptr ? 1.f / (1.f + expf(-g0)) : 1.f;
    // weight 0 is for records that were not written (maximum -inf, sum 0); a NaN or infinite score makes the sum NaN
    if (lane < 32) ws[wave][lane] = m == -INFINITY && l == 0.f ? 0.f : e / den * gh;
  }
  lds_barrier();
  if (k < nt) {
    f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
    auto add = [&](const f32x4& v, int s) {
      const float w = s < nsplit ? ws[k][s] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] += w != 0.f ? w * v[i] : 0.f;             // (w 0: nothing, or nothing written)
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) add(x[u], u);
    for (int s = AHEAD; s < nsplit; s += 8) {
      f32x4 z[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) z[u] = *reinterpret_cast<const f32x4*>(pr + (size_t)min(s + u, nsplit - 1) * C);
#pragma unroll
      for (int u = 0; u < 8; ++u) add(z[u], s + u);
    }
    stf4(&lat[k][c], y);
  }
  lds_barrier();
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[kk], *reinterpret_cast<const bf16x8*>(&lat[li][32 * (kk0 + kk) + 8 * g]), acc,
                                                  0, 0, 0);
  // acc[i] = out[token li][value column v0 + 16 cb + 4 g + i], this wave's share of k
  if constexpr (KS > 1) {
    *reinterpret_cast<f32x4*>(part[wave / CB][cb][lane]) = acc;
    lds_barrier();
    if (wave >= CB) return;
#pragma unroll
    for (int x = 1; x < KS; ++x) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(part[x][cb][lane]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += y[i];
    }
  }
  if (li < nt) stf4(out + ((size_t)(t0 + li) * H + hd) * V + v0 + 16 * cb + 4 * g, acc);
}

}  // namespace k8sllm

using namespace k8sllm;

// Whether the kernels take these sizes.
extern "C" int k8s_latent_token_ok(int C, int R, int Dn, int V) { return C == 512 && R == 64 && Dn % 8 == 0 && V == 128; }

// out [T][H][V] bf16; pacc [T][HP][nsplit][C], pml [T][HP][nsplit][2] fp32 workspaces with HP = H rounded up to 16.
extern "C" int k8s_latent_token(void* out, float* pacc, float* pml, const void* q_abs, const void* q, const void* cache,
                                const void* uv, const int* block_tables, int max_blocks, const int* tok_seq,
                                const int* positions, int T, int C, int R, int H, int Dn, int V, int window, float scale,
                                int bs, int nsplit, const float* sinks, const void* gate, long ldg, hipStream_t s) {
  if (T <= 0) return 0;
  if (!k8s_latent_token_ok(C, R, Dn, V) || H <= 0 || bs <= 0 || nsplit < 1 || nsplit > 32 || T > (1 << 20)) return -1;
  if (gate != nullptr && ldg < H) return -1;
  if ((((uintptr_t)q_abs | (uintptr_t)q | (uintptr_t)cache | (uintptr_t)uv | (uintptr_t)out | (uintptr_t)pacc) & 15) != 0)
    return -1;
  const int hg = (H + 15) / 16;
  constexpr int LDS = 64 * (576 + 8) * 2 + 16 * 72 * 2 + 64 * 4;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(latent_token_kernel<512, 64>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  latent_token_kernel<512, 64><<<dim3(T, hg, nsplit), 256, LDS, s>>>(pacc, pml, (const bf16_t*)q_abs, (const bf16_t*)q,
                                                                     (const bf16_t*)cache, block_tables, max_blocks, tok_seq,
                                                                     positions, H, Dn, window, scale, bs, nsplit);
  // few heads and tokens: a quarter of a head's value columns a workgroup.  A compute unit takes the weights of 128 columns, rows of 64
  // bytes to an instruction, in about 4 us whoever else is idle; the splits' sums are read four times as often, from L2
  const int groups = (T + 3) / 4;
#define K8S_LO(CB)                                                                                                                  \
  latent_out_kernel<512, 128, CB><<<dim3(H * (8 / CB), groups), 512, 0, s>>>((bf16_t*)out, pacc, pml, (const bf16_t*)uv, T, H, hg * 16, \
                                                                             nsplit, sinks, (const bf16_t*)gate, ldg)
  if (H * groups < 128) K8S_LO(2);
  else K8S_LO(8);
#undef K8S_LO
  return (int)hipGetLastError();
}
