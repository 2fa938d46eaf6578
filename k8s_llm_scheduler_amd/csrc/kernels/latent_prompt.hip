// Latent attention of prompts with the keys and values written out.
//
// The cache holds one low-rank row per token, [normed latent (C) | rotated key part (R)].  Attending it as it is stored
// (mixers.hip) costs C + R multiply-adds per query, key and head for the score and C for the value; a head's own key and
// value take DN + R and DV.  For a portion of n tokens of a sequence whose visible keys are K rows, writing out every visible
// row's keys and values once, c [W_uk | W_uv]^T, costs K C (DN + DV) per head (the absorbed form spends n C (DN + DV) on
// queries and outputs instead) and saves about n K (2 C - DN - DV): at C = 512, DN = DV = 128 it pays from n = 170 on
// whatever is cached already, and always where nothing is.
//
// Three steps: latent_keys_kernel lists the cache slots of the rows that the batch's tokens see, compactly, sequence after
// sequence, with the row tiles of the product that follows; the grouped GEMM (stream32.hip) gathers those latents and writes
// [keys (DN) | values (DV)] per head; the kernels below attend them.
#include "common.h"

namespace k8sllm {

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// First visible key of a sequence's portion and the number of visible rows; idle and empty sequences have none.
__device__ __forceinline__ int latent_span(const int* cu_q, const int* positions, int s, int window, int& lo) {
  const int a = cu_q[s], b = cu_q[s + 1];
  lo = 0;
  if (b <= a || positions[a] < 0) return 0;
  const int p = positions[a];
  lo = window > 0 ? max(0, p - window + 1) : 0;
  return p + (b - a) - lo;
}

// One workgroup per sequence: rows[kbase[s] + i] = cache slot of the sequence's key lo + i; tiles (0, first row, rows) of at
// most 64 rows each, the entries behind the last one (-1, 0, 0); seg = (0, rows of all sequences).
__global__ __launch_bounds__(256) void latent_keys_kernel(int* __restrict__ rows, int* __restrict__ kbase,
                                                          int* __restrict__ tiles, int* __restrict__ seg,
                                                          const int* __restrict__ cu_q,
                                                          const int* __restrict__ positions,
                                                          const int* __restrict__ block_tables, int max_blocks, int nseq,
                                                          int window, int bs, int cap, int ntiles) {
  __shared__ float red[16];        // the sums are whole numbers below 2^24
  const int s = blockIdx.x;
  float nr = 0.f, nt = 0.f;
  int lo;
  for (int i = threadIdx.x; i < s; i += blockDim.x) {
    const int n = latent_span(cu_q, positions, i, window, lo);
    nr += (float)n;
    nt += (float)((n + 63) / 64);
  }
  const int base = (int)block_sum(nr, red), tile0 = (int)block_sum(nt, red);
  const int n = min(latent_span(cu_q, positions, s, window, lo), cap - base);
  if (threadIdx.x == 0) {
    kbase[s] = base;
    if (s == nseq - 1) {
      seg[0] = 0;
      seg[1] = base + max(n, 0);
    }
  }
  const int* btr = block_tables + (size_t)s * max_blocks;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int key = lo + i, page = key / bs;
    rows[base + i] = btr[page] * bs + (key - page * bs);
  }
  const int mine = (max(n, 0) + 63) / 64, stop = s == nseq - 1 ? ntiles : min(ntiles, tile0 + mine);
  for (int i = threadIdx.x; tile0 + i < stop; i += blockDim.x) {
    int* t = tiles + 3 * (tile0 + i);
    t[0] = i < mine ? 0 : -1;
    t[1] = i < mine ? base + 64 * i : 0;
    t[2] = i < mine ? min(64, n - 64 * i) : 0;
  }
}

__device__ __forceinline__ float latent_gate(const bf16_t* gate, long ldg, int t, int hd) {
  return gate != nullptr ? 1.f / (1.f + expf(-bf2f(gate[(size_t)t * ldg + hd]))) : 1.f;
}

// bf16.  S^T = K Q^T with a head's queries as the 16 columns of a tile, O += P V through the transposing LDS read, softmax in
// fp32 with the weights rounded to bf16 for the product (as the absorbed kernel has them).  A workgroup takes 64 NCB tokens
// of one head: 8 waves in two groups that own the same tokens (a wave NCB blocks of 16) and take the first and the second
// half of every 64-key step with a running softmax of their own; two LDS buffers, the next step stored and the one after
// next loaded into registers under this one's products, its rows' slots a step earlier still; scores in base 2, no mask
// arithmetic on slices that every column sees, accumulators rescaled only when a maximum moved.  Workgroups of one head
// follow each other at a distance of H, so with H a multiple of 8 a head's keys stay in one XCD's L2.
// 2048 tokens, 16 heads, a window of 1024: 50 us, 330 TFLOP/s, and 35 us for the keys and values (absorbed: 317 us and 66 us
// for its two products).  Bound by the LDS reads of two waves per SIMD and the softmax between the products.
template <int DN, int R, int DV, int NCB>
__global__ __launch_bounds__(512) void latent_prompt_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ kv, const int* __restrict__ rows, const int* __restrict__ kbase,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, int C, const int* __restrict__ cu_q,
    const int* __restrict__ positions, int H, int window, float scale, const float* __restrict__ sinks,
    const bf16_t* __restrict__ gate, long ldg) {
  constexpr int DK = DN + R, NKK = DK / 32, NVB = DV / 16, KT = 64;
  constexpr int ROWK = (DK + 8) * 2, ROWV = (DV + 8) * 2, BUF = KT * (ROWK + ROWV);   // LDS bytes
  constexpr int CN = DN / 8, CK = DK / 8, CV = DV / 8, NST = (CK + CV + 7) / 8;      // 16-byte pieces; per thread
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(16))) char smem_p[];
  const int hd = blockIdx.x, seq = blockIdx.z;
  const int tid = threadIdx.x, wave = (tid >> 6) & 3, grp = tid >> 8, lane = tid & 63, li = lane & 15, g4 = lane >> 4;
  constexpr int TPB = 64 * NCB;
  const int tile = gridDim.y - 1 - blockIdx.y;               // the tiles with most keys first
  const int tq0 = cu_q[seq] + tile * TPB, tend = cu_q[seq + 1];
  if (tq0 >= tend) return;
  const int p_first = positions[tq0], p_seq = p_first - tile * TPB;
  const int nval = min(TPB, tend - tq0);
  if (p_first < 0) {   // idle rows: defined output
    for (int i = tid; i < nval * DV; i += 512) out[((size_t)(tq0 + i / DV) * H + hd) * DV + i % DV] = 0;
    return;
  }
  const int p_last = p_first + nval - 1;
  auto lo_of = [&](int p) { return window > 0 ? max(0, p - window + 1) : 0; };
  const int lo_min = lo_of(p_first), nkeys = p_last + 1 - lo_min, nsteps = (nkeys + KT - 1) / KT;
  const int row0 = kbase[seq] + lo_min - lo_of(p_seq);       // compact row of key lo_min
  const size_t ldkv = (size_t)H * (DN + DV), kvo = (size_t)hd * (DN + DV);
  const int L = C + R;
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  int c_p[NCB], c_lo[NCB];
  bf16x8 qf[NCB][NKK];
  int w_pmin = 0x7fffffff, w_pmax = -1;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const int toff = (wave * NCB + cb) * 16 + li;
    const bool ok = toff < nval;
    c_p[cb] = ok ? p_first + toff : -1;
    c_lo[cb] = ok ? lo_of(c_p[cb]) : 0;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      u32x4 v = zero;
      if (ok) v = *reinterpret_cast<const u32x4*>(q + ((size_t)(tq0 + toff) * H + hd) * DK + 32 * kk + 8 * g4);
      qf[cb][kk] = __builtin_bit_cast(bf16x8, v);
    }
    const int t_lo = (wave * NCB + cb) * 16, t_hi = min(t_lo + 16, nval) - 1;
    if (t_lo < nval) {
      w_pmin = min(w_pmin, p_first + t_lo);
      w_pmax = max(w_pmax, p_first + t_hi);
    }
  }
  const bool w_any = w_pmax >= 0;
  const int w_lo = w_any ? lo_of(w_pmin) : 0, w_hi_lo = w_any ? lo_of(w_pmax) : 0;   // first key any / every column sees
  const bool with_sink = sinks != nullptr && grp == 0;
  const float sc2 = scale * LOG2E;
  f32x4 o[NCB][NVB];
  float m_run[NCB], l_run[NCB];                  // l_run: this lane's keys only
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    m_run[cb] = with_sink ? sinks[hd] * LOG2E : -INFINITY;
    l_run[cb] = with_sink && g4 == 0 ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NVB; ++n) o[cb][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int qd = li >> 2, pd = li & 3;
  // staging: thread -> row tid / 8 of the step, pieces tid % 8 + 8 i of [key | rotated part | value]
  const int sr = tid >> 3, sc = tid & 7;
  u32x4 pre[NST];
  auto slot_of = [&](int step) -> int {
    const int u = step * KT + sr;
    return u < nkeys ? rows[row0 + u] : -1;
  };
  auto stage_load = [&](int step, int slot) {
    const bf16_t* kr = kv + (size_t)(row0 + step * KT + sr) * ldkv + kvo;
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = sc + 8 * i;
      u32x4 v = zero;
      if (slot >= 0 && c < CK + CV)
        v = c < CN ? *reinterpret_cast<const u32x4*>(kr + 8 * c)
          : c < CK ? *reinterpret_cast<const u32x4*>(cache + (size_t)slot * L + C + 8 * (c - CN))
                   : *reinterpret_cast<const u32x4*>(kr + DN + 8 * (c - CK));
      pre[i] = v;
    }
  };
  auto stage_store = [&](char* buf) {
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = sc + 8 * i;
      if (c < CK) *reinterpret_cast<u32x4*>(buf + sr * ROWK + 16 * c) = pre[i];
      else if (c < CK + CV) *reinterpret_cast<u32x4*>(buf + KT * ROWK + sr * ROWV + 16 * (c - CK)) = pre[i];
    }
  };
  stage_load(0, slot_of(0));
  stage_store(smem_p);
  int slot = -1;
  if (nsteps > 1) stage_load(1, slot_of(1));
  if (nsteps > 2) slot = slot_of(2);
  __syncthreads();
  for (int step = 0; step < nsteps; ++step) {
    char* buf = smem_p + (step & 1) * BUF;
    if (step + 1 < nsteps) {
      stage_store(smem_p + ((step + 1) & 1) * BUF);
      if (step + 2 < nsteps) {
        stage_load(step + 2, slot);
        slot = step + 3 < nsteps ? slot_of(step + 3) : -1;
      }
    }
    const int j0 = lo_min + step * KT + 32 * grp;          // this group's slice: keys j0 .. j0 + 31
    if (w_any && j0 <= w_pmax && j0 + 31 >= w_lo) {
      const char* klds = buf + 32 * grp * ROWK;
      const char* vlds = buf + KT * ROWK + 32 * grp * ROWV;
      f32x4 sacc[NCB][2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) sacc[cb][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
          const bf16x8 ka = *reinterpret_cast<const bf16x8*>(klds + (16 * m + li) * ROWK + 64 * kk + 16 * g4);
#pragma unroll
          for (int cb = 0; cb < NCB; ++cb)
            sacc[cb][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[cb][kk], sacc[cb][m], 0, 0, 0);
        }
      }   // sacc[cb][m][i] = S[key j0 + 16 m + 4 g4 + i][column li of block cb]
      const bool all_seen = j0 >= w_hi_lo && j0 + 31 <= w_pmin;
      bf16x8 pa[NCB];            // slot j < 4: key 4 g4 + j; slot j >= 4: key 16 + 4 g4 + (j - 4)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) sacc[cb][m][i] *= sc2;
        if (!all_seen) {
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = j0 + 16 * m + 4 * g4 + i;
              if (j > c_p[cb] || j < c_lo[cb]) sacc[cb][m][i] = -INFINITY;
            }
        }
        float tmax = fmaxf(fmaxf(fmaxf(sacc[cb][0][0], sacc[cb][0][1]), fmaxf(sacc[cb][0][2], sacc[cb][0][3])),
                           fmaxf(fmaxf(sacc[cb][1][0], sacc[cb][1][1]), fmaxf(sacc[cb][1][2], sacc[cb][1][3])));
        tmax = lane_max<16>(tmax);
        tmax = lane_max<32>(tmax);
        if (__any(tmax > m_run[cb])) {
          const float m_new = fmaxf(m_run[cb], tmax);
          const float alpha = m_run[cb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[cb] - m_new);
          m_run[cb] = m_new;
          l_run[cb] *= alpha;
          float a_i[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) a_i[i] = __shfl(alpha, g4 * 4 + i, WAVE);
#pragma unroll
          for (int n = 0; n < NVB; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[cb][n][i] *= a_i[i];
        }
        const float m_ref = m_run[cb] == -INFINITY ? 0.f : m_run[cb];      // a column that has seen nothing yet
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sacc[cb][m][i] = __builtin_amdgcn_exp2f(sacc[cb][m][i] - m_ref);
            l_run[cb] += sacc[cb][m][i];
          }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pa[cb][j] = (__bf16)sacc[cb][0][j];
          pa[cb][4 + j] = (__bf16)sacc[cb][1][j];
        }
      }
      const int r0 = 4 * g4 + qd, r1 = r0 + 16;
#pragma unroll
      for (int n = 0; n < NVB; ++n) {
        const int col = 16 * n + 4 * pd;
        const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vlds + r0 * ROWV + 2 * col));
        const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vlds + r1 * ROWV + 2 * col));
        bf16x8 vb;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vb[j] = v0[j]; vb[4 + j] = v1[j]; }
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb)
          o[cb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[cb], vb, o[cb][n], 0, 0, 0);
      }
    }
    __syncthreads();          // this step's fragments have been read, the next step is staged
  }
  // o[cb][n][i] = O[column 4 g4 + i][d 16 n + li]; m_run, l_run belong to column li.  Group 1 leaves its part in LDS.
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    l_run[cb] = lane_sum<16>(l_run[cb]);
    l_run[cb] = lane_sum<32>(l_run[cb]);
  }
  float* mo = reinterpret_cast<float*>(smem_p) + (size_t)wave * 64 * NCB * (4 * NVB + 2);   // [NCB (4 NVB + 2)][64 lanes]
  if (grp == 1) {
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      float* b = mo + cb * (4 * NVB + 2) * 64 + lane;
#pragma unroll
      for (int n = 0; n < NVB; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) b[(4 * n + i) * 64] = o[cb][n][i];
      b[4 * NVB * 64] = m_run[cb];
      b[(4 * NVB + 1) * 64] = l_run[cb];
    }
  }
  __syncthreads();
  if (grp == 1) return;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const float* b = mo + cb * (4 * NVB + 2) * 64 + lane;
    const float m1 = b[4 * NVB * 64], M = fmaxf(m_run[cb], m1);
    const float f0 = m_run[cb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[cb] - M);
    const float f1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - M);
    const float inv = 1.f / (l_run[cb] * f0 + b[(4 * NVB + 1) * 64] * f1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 4 * g4 + i;
      const float w0 = __shfl(f0 * inv, c, WAVE), w1 = __shfl(f1 * inv, c, WAVE);
      const int toff = (wave * NCB + cb) * 16 + c;
      if (toff >= nval) continue;
      const int t = tq0 + toff;
      const float s = latent_gate(gate, ldg, t, hd);
#pragma unroll
      for (int n = 0; n < NVB; ++n)
        out[((size_t)t * H + hd) * DV + 16 * n + li] = f2bf((o[cb][n][i] * w0 + b[(4 * n + i) * 64] * w1) * s);
    }
  }
}

// fp32, every product and sum in fp32 (v_mfma_f32_16x16x4_f32).  A workgroup takes 64 tokens of one head, a wave 16 of them;
// 32-key steps staged through LDS.  S^T = K Q^T leaves a lane the scores of the keys 16 m + 4 g + i of its token; O^T = V^T P
// takes them as the B operand of the instruction (m, i) where they are, so nothing is exchanged but the maxima and sums.
// DK = DN + R and DV multiples of 16.  A score is four sums of every fourth dimension: in one, 48 instructions long, it was the largest
// part of the result's error (2-norm against 64 bits 4.0 - 4.9e-7, so 2.7 - 3.5e-7; 45 -> 47 us).  333 tokens, 16 heads: 47 us (absorbed 104
// in latent_f32.hip); six token tiles of 16 heads leave most of the chip idle.
template <int DN, int R, int DV>
__global__ __launch_bounds__(256) void latent_prompt_f32_kernel(
    float* __restrict__ out, const float* __restrict__ kv, const int* __restrict__ rows, const int* __restrict__ kbase,
    const float* __restrict__ q, const float* __restrict__ cache, int C, const int* __restrict__ cu_q,
    const int* __restrict__ positions, int H, int window, float scale, const float* __restrict__ sinks,
    const float* __restrict__ gate, long ldg) {
  constexpr int DK = DN + R, NK4 = DK / 16, NVB = DV / 16, KT = 32, LDK = DK + 4, LDV = DV + 4;
  constexpr int CN = DN / 4, CK = DK / 4, CV = DV / 4, NST = (CK + CV + 7) / 8;      // 16-byte pieces; per thread
  __shared__ __attribute__((aligned(16))) float ks[KT][LDK];
  __shared__ __attribute__((aligned(16))) float vs[KT][LDV];
  const int hd = blockIdx.x, seq = blockIdx.z, tile = gridDim.y - 1 - blockIdx.y;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int tq0 = cu_q[seq] + tile * 64, tend = cu_q[seq + 1];
  if (tq0 >= tend) return;
  const int p_first = positions[tq0], p_seq = p_first - tile * 64;
  const int nval = min(64, tend - tq0);
  if (p_first < 0) {   // idle rows: defined output
    for (int i = tid; i < nval * DV; i += 256) out[((size_t)(tq0 + i / DV) * H + hd) * DV + i % DV] = 0.f;
    return;
  }
  const int p_last = p_first + nval - 1;
  auto lo_of = [&](int p) { return window > 0 ? max(0, p - window + 1) : 0; };
  const int lo_min = lo_of(p_first), nkeys = p_last + 1 - lo_min, nsteps = (nkeys + KT - 1) / KT;
  const int row0 = kbase[seq] + lo_min - lo_of(p_seq);
  const size_t ldkv = (size_t)H * (DN + DV), kvo = (size_t)hd * (DN + DV);
  const int L = C + R, toff = 16 * wave + li;
  const bool ok = toff < nval;
  const int p = ok ? p_first + toff : -1, lo = ok ? lo_of(p) : 0;
  const int w_first = p_first + 16 * wave, w_last = min(w_first + 15, p_last);   // this wave's tokens
  const bool w_any = 16 * wave < nval;
  const int w_lo = w_any ? lo_of(w_first) : 0;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 qf[NK4];               // B operand of instruction (j, i): q[16 j + 4 g + i]
#pragma unroll
  for (int j = 0; j < NK4; ++j)
    qf[j] = ok ? *reinterpret_cast<const f32x4*>(q + ((size_t)(tq0 + toff) * H + hd) * DK + 16 * j + 4 * g) : zero;
  f32x4 o[NVB];                // o[n][i] = O[d 16 n + 4 g + i][token li]
#pragma unroll
  for (int n = 0; n < NVB; ++n) o[n] = zero;
  float m_run = sinks != nullptr ? sinks[hd] : -INFINITY, l_run = sinks != nullptr && g == 0 ? 1.f : 0.f;
  const int sr = tid >> 3, sc = tid & 7;
  f32x4 pre[NST];
  auto stage_load = [&](int step) {
    const int u = step * KT + sr;
    const int slot = u < nkeys ? rows[row0 + u] : -1;
    const float* kr = kv + (size_t)(row0 + u) * ldkv + kvo;
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = sc + 8 * i;
      f32x4 v = zero;
      if (slot >= 0 && c < CK + CV)
        v = c < CN ? *reinterpret_cast<const f32x4*>(kr + 4 * c)
          : c < CK ? *reinterpret_cast<const f32x4*>(cache + (size_t)slot * L + C + 4 * (c - CN))
                   : *reinterpret_cast<const f32x4*>(kr + DN + 4 * (c - CK));
      pre[i] = v;
    }
  };
  stage_load(0);
  for (int step = 0; step < nsteps; ++step) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = sc + 8 * i;
      if (c < CK) *reinterpret_cast<f32x4*>(&ks[sr][4 * c]) = pre[i];
      else if (c < CK + CV) *reinterpret_cast<f32x4*>(&vs[sr][4 * (c - CK)]) = pre[i];
    }
    __syncthreads();
    if (step + 1 < nsteps) stage_load(step + 1);
    const int j0 = lo_min + step * KT;
    if (!w_any || j0 > w_last || j0 + KT - 1 < w_lo) continue;
    f32x4 s[2];                    // s[m][i] = score of key j0 + 16 m + 4 g + i for token li
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      f32x4 part[4] = {zero, zero, zero, zero};
#pragma unroll
      for (int j = 0; j < NK4; ++j) {
        const f32x4 kf = *reinterpret_cast<const f32x4*>(&ks[16 * m + li][16 * j + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], qf[j][i], part[i], 0, 0, 0);
      }
      s[m] = (part[0] + part[1]) + (part[2] + part[3]);
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = j0 + 16 * m + 4 * g + i;
        s[m][i] = key <= p && key >= lo ? s[m][i] * scale : -INFINITY;
        tmax = fmaxf(tmax, s[m][i]);
      }
    tmax = lane_max<16>(tmax);
    tmax = lane_max<32>(tmax);
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = m_run == -INFINITY ? 0.f : expf(m_run - m_new);
    const float m_ref = m_new == -INFINITY ? 0.f : m_new;      // a token that has seen nothing yet
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[m][i] = expf(s[m][i] - m_ref);
        l_run += s[m][i];
      }
#pragma unroll
    for (int n = 0; n < NVB; ++n) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[n][i] *= alpha;
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[16 * m + 4 * g + i][16 * n + li], s[m][i], o[n], 0, 0, 0);
    }
  }
  if (!ok) return;
  l_run = lane_sum<16>(l_run);
  l_run = lane_sum<32>(l_run);
  float f = 1.f / l_run;
  if (gate != nullptr) f /= 1.f + expf(-gate[(size_t)(tq0 + toff) * ldg + hd]);
#pragma unroll
  for (int n = 0; n < NVB; ++n) {
    f32x4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = o[n][i] * f;
    *reinterpret_cast<f32x4*>(out + ((size_t)(tq0 + toff) * H + hd) * DV + 16 * n + 4 * g) = y;
  }
}

}  // namespace k8sllm

using namespace k8sllm;

// Whether the kernels take these sizes.
extern "C" int k8s_latent_prompt_ok(int C, int R, int Dn, int V) { return C % 8 == 0 && Dn == 128 && R == 64 && V == 128; }

// rows [cap], kbase [nseq], tiles [ntiles][3], seg [2]; cap and ntiles bound the batch's visible rows and their tiles.
extern "C" int k8s_latent_keys(int* rows, int* kbase, int* tiles, int* seg, const int* cu_q, const int* positions,
                               const int* block_tables, int max_blocks, int nseq, int window, int bs, int cap, int ntiles,
                               hipStream_t s) {
  if (nseq <= 0) return 0;
  if (bs <= 0 || cap <= 0 || cap >= (1 << 24) || ntiles < cap / 64 + nseq) return -1;
  latent_keys_kernel<<<nseq, 256, 0, s>>>(rows, kbase, tiles, seg, cu_q, positions, block_tables, max_blocks, nseq, window, bs, cap,
                                          ntiles);
  return (int)hipGetLastError();
}

// kv [rows][H][Dn + V]: the listed rows' keys and values; out [T][H][V].
extern "C" int k8s_latent_prompt(void* out, const void* kv, const int* rows, const int* kbase, const void* q,
                                 const void* cache, int C, int R, int Dn, int V, const int* cu_q, const int* positions,
                                 int nseq, int max_qlen, int H, int window, float scale, const float* sinks,
                                 const void* gate, long ldg, int f32, hipStream_t s) {
  if (nseq <= 0 || max_qlen <= 0) return 0;
  if (!k8s_latent_prompt_ok(C, R, Dn, V) || H <= 0 || nseq > 65535 || (gate != nullptr && ldg < H)) return -1;
  if ((((uintptr_t)q | (uintptr_t)kv | (uintptr_t)cache | (uintptr_t)out) & 15) != 0) return -1;
  if (f32) {
    const dim3 grid(H, (max_qlen + 63) / 64, nseq);
    if (grid.y > 65535) return -2;
    latent_prompt_f32_kernel<128, 64, 128><<<grid, 256, 0, s>>>((float*)out, (const float*)kv, rows, kbase, (const float*)q,
                                                                (const float*)cache, C, cu_q, positions, H, window, scale,
                                                                sinks, (const float*)gate, ldg);
    return (int)hipGetLastError();
  }
#define K8S_LP(NCB)                                                                                                      \
  do {                                                                                                                   \
    constexpr int BUF = 64 * ((192 + 8) * 2 + (128 + 8) * 2), MO = 4 * 64 * NCB * (4 * 8 + 2) * 4;                       \
    constexpr int LDS = 2 * BUF > MO ? 2 * BUF : MO;                                                                     \
    const dim3 grid(H, (max_qlen + 64 * NCB - 1) / (64 * NCB), nseq);                                                    \
    if (grid.y > 65535) return -2;                                                                                       \
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(latent_prompt_kernel<128, 64, 128, NCB>),     \
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS);                           \
    if (e != hipSuccess) return (int)e;                                                                                  \
    latent_prompt_kernel<128, 64, 128, NCB><<<grid, 512, LDS, s>>>(                                                      \
        (bf16_t*)out, (const bf16_t*)kv, rows, kbase, (const bf16_t*)q, (const bf16_t*)cache, C, cu_q, positions, H,     \
        window, scale, sinks, (const bf16_t*)gate, ldg);                                                                 \
  } while (0)
  if ((long)H * ((max_qlen + 127) / 128) * nseq >= 256) K8S_LP(2);
  else K8S_LP(1);
#undef K8S_LP
  return (int)hipGetLastError();
}
