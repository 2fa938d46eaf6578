// K6: causal prefill flash attention over the PAGED KV cache, MFMA bf16 (gfx950).
//
// Reading K/V through the block table (instead of from the chunk's own q/k/v) makes the same
// kernel serve plain prefill, chunked prefill and prefix-cached prompts: query i of sequence s
// sits at absolute position ctx_s - qlen_s + i and attends keys [0, pos].
//
// GQA packing: a wave has 16 RB (query, head) rows, a workgroup those of NW / KS waves = QT consecutive queries x the G query
// heads that share ONE kv head (G = nq / nkv), so every K/V tile is fetched once per group instead of once per query head, and
// the causal key range of a workgroup ends at its last query.  Row r of the workgroup is query tile * QT + r / G, head kvh * G +
// r % G.  KS 2: half of the waves takes every other tile of the same rows' keys; their sums meet at the end.
//
// Structure:
//  * "swapped" QK^T: S^T = K . Q^T with v_mfma_f32_16x16x32_bf16, so each lane ends up holding 16 scores of ONE query row (row =
//    lane & 15) and the probabilities feed the P.V MFMA as its B operand straight from registers (the key order inside a 32-key
//    step is permuted identically on the V side, see below), whose result O^T has a query row in the same lanes.
//  * V tiles (64 keys x 128 d) are staged in LDS with an XOR swizzle and read with the gfx950 transposing read
//    ds_read_b64_tr_b16, which delivers 4 keys of one d column per lane -- exactly the A-operand layout.
//  * K and V go through registers into two swizzled LDS images each: the tile after next is on its way, the next one is written,
//    one barrier a tile that waits for LDS only.
//  * 32 rows a wave (RB 2) read each K and V fragment for two products: at 16 rows a wave's LDS reads take twice the time of its
//    products.
//  * online softmax in the log2 domain: one fma (scale and maximum), maximum, power and addition a score; the lanes of a row meet,
//    and the sums are rescaled, only in tiles where a row of the block has outgrown its maximum; masks only where a tile crosses
//    the wave's diagonal.  (A reference up to 2^12 below the maximum would spare most of the rest; the largest weight, 1 here, would
//    then be rounded to bf16: 3 - 8 % more error against 64 bits.)
//  * longest workgroups first, so that the last round is of short ones.
// What bounds it now: two waves a SIMD, in step between the barriers, each with its products, LDS reads and softmax in turn; at
// long prompts 35 % of the matrix cores' rate.  Tried: waves of a SIMD half a tile apart with two barriers a tile (251 us against
// 230 at 3413 tokens, without the running maximum), 128 rows of 4 waves (256 us), one branch for both blocks of rows (272 us
// against 266).
#include "common.h"

#define K8S_CHK_THIS_UNIT 5

namespace k8sllm {

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

__device__ __forceinline__ int v_swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// Over the four lanes that share a column of a 16 x 16 product (l, l ^ 16, l ^ 32, l ^ 48), in all of them, by register moves: odd rows of 16 lanes of one copy against
// even ones of the other, then halves.  (In asm with its wait states: the builtins hand back the first of the two registers twice.)
template <typename F>
__device__ __forceinline__ float row_join(float v, F f) {
  float x = v, y = v;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
  x = y = f(x, y);
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
  return f(x, y);
}
__device__ __forceinline__ float row_max(float v) {
  return row_join(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float row_sum(float v) {
  return row_join(v, [](float a, float b) { return a + b; });
}

template <int G, int RB, int NW, int KS>
__global__ void __launch_bounds__(64 * NW, 2) paged_prefill_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int* __restrict__ cu_q, const int* __restrict__ context_lens,
    const int* __restrict__ block_tables, float scale_log2, int nq, int nkv, int block_size, int max_blocks, int tiles) {
  constexpr int D = 128;
  constexpr int KT = 64;                // keys per tile
  constexpr int ST = KS * KT;           // keys staged at once: a tile for each share of the waves
  constexpr int NT = 64 * NW;           // threads
  constexpr int CPT = ST * D / 8 / NT;  // 16-byte chunks of what is staged per thread (K and V each)
  constexpr int RW = NW / KS;           // waves of a share
  constexpr int QT = 16 * RB * RW / G;  // queries per workgroup
  static_assert(16 * RB % G == 0 || G % (16 * RB) == 0, "a wave's rows are whole queries or part of one");
  __shared__ __attribute__((aligned(16))) char klds[2][ST * D * 2];
  __shared__ __attribute__((aligned(16))) char vlds[2][ST * D * 2];

  // the longest workgroups first; those of a kv head follow each other at a stride of the heads
  const int s = blockIdx.z, kvh = blockIdx.x % nkv, tile = tiles - 1 - blockIdx.x / nkv;
  const int q0 = cu_q[s], qlen = cu_q[s + 1] - q0;
  if (tile * QT >= qlen) return;
  int ctx = context_lens[s];
  K8S_CHECK_MAX(ctx, max_blocks * block_size, K8S_CHK_CTX);
  const int qstart = ctx - qlen;  // absolute position of query 0
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wid = wave % RW, share = wave / RW;   // which rows, which tile of those staged
  const int g = lane >> 4, li = lane & 15;
  const int* bt = block_tables + (size_t)s * max_blocks;
  const int last_row = min(tile * QT + QT - 1, qlen - 1);
  const int kv_end = qstart + last_row + 1;  // keys needed by this workgroup
  const int ntiles = (kv_end + ST - 1) / ST;

  // Tile staging: thread tid fetches chunks idx = tid + NT c (key row idx/16, 16-byte column chunk idx%16) of K and V into
  // registers while tiles before are computed.  Rows past the context lie in the last key's block (finite or not: K's scores are
  // masked), V is zeroed there (P is 0, V must be finite).  The block ids of a tile are requested a tile before its K/V: otherwise
  // every prefetch is two dependent round trips.  Where a row is in its block is carried from tile to tile: the division by the
  // block size was half of the loop's vector work.
  u32x4 kn[CPT], vn[CPT];
  int nbt[CPT], nbv[CPT], wof[CPT], wov[CPT];    // block ids of the next K and V tile's rows, rows in the blocks
  int ib[CPT], io[CPT];                          // block table position and row in the block of the next ids
  const int lastb = (ctx - 1) / block_size, stepb = ST / block_size, stepo = ST - stepb * block_size;
  const unsigned row_bytes = (unsigned)nkv * D * 2;
  const char* kp = reinterpret_cast<const char*>(k_cache) + (kvh * D + tid % (D / 8) * 8) * 2;
  const char* vp = reinterpret_cast<const char*>(v_cache) + (kvh * D + tid % (D / 8) * 8) * 2;
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int r = (tid + NT * c) / (D / 8);
    ib[c] = r / block_size;
    io[c] = r - ib[c] * block_size;
  }
  auto ids = [&]() {                             // of the next tile
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      nbt[c] = bt[min(ib[c], lastb)];
      K8S_CHECK_RANGE(nbt[c], 0, K8S_CHK_BLOCK, 0);
      wof[c] = io[c];
      ib[c] += stepb;
      io[c] += stepo;
      const bool wrap = io[c] >= block_size;
      io[c] -= wrap ? block_size : 0;
      ib[c] += wrap;
    }
  };
  auto keep = [&]() {                            // K's ids for V, a tile later
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      nbv[c] = nbt[c];
      wov[c] = wof[c];
    }
  };
  auto fetch_k = [&]() {
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      kn[c] = *reinterpret_cast<const u32x4*>(kp + (size_t)(unsigned)(nbt[c] * block_size + wof[c]) * row_bytes);
  };
  auto fetch_v = [&]() {
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      vn[c] = *reinterpret_cast<const u32x4*>(vp + (size_t)(unsigned)(nbv[c] * block_size + wov[c]) * row_bytes);
  };
  auto mask_v = [&](int t) {                     // tile t's, ahead of its staging
    if (t * ST + ST <= ctx) return;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      if (t * ST + (tid + NT * c) / (D / 8) >= ctx) vn[c] = u32x4{0u, 0u, 0u, 0u};
  };
  auto stage_k = [&](int buf) {   // both images swizzled: 16-byte chunk ch of row r at ch ^ swz(r)
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int kr = (tid + NT * c) / (D / 8), ch = (tid + NT * c) % (D / 8);
      *reinterpret_cast<u32x4*>(klds[buf] + kr * (D * 2) + 16 * (ch ^ (kr & 15))) = kn[c];
    }
  };
  auto stage_v = [&](int buf) {
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int kr = (tid + NT * c) / (D / 8), ch = (tid + NT * c) % (D / 8);
      *reinterpret_cast<u32x4*>(vlds[buf] + kr * (D * 2) + 16 * (ch ^ v_swz(kr))) = vn[c];
    }
  };
  ids();
  fetch_k();
  keep();

  // my (query, head) rows (B operand columns / softmax rows)
  bf16x8 qf[RB][D / 32];
  int qpos[RB];
  // (a negative scale: of the negated queries; 0, which the masked scores could not take: of zeros)
  const uint32_t flip = scale_log2 < 0.f ? 0x80008000u : 0u, live = scale_log2 == 0.f ? 0u : ~0u;
  const float scale = scale_log2 == 0.f ? 1.f : fabsf(scale_log2);
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const int wr = (wid * RB + b) * 16 + li;
    const int row = min(tile * QT + wr / G, qlen - 1), head = kvh * G + wr % G;   // (padding rows: a valid query)
    qpos[b] = qstart + row;
    const u32x4* qp = reinterpret_cast<const u32x4*>(q + ((size_t)(q0 + row) * nq + head) * D);
#pragma unroll
    for (int kk = 0; kk < D / 32; ++kk) {
      u32x4 v = qp[kk * 4 + g];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (v[e] ^ flip) & live;
      qf[b][kk] = __builtin_bit_cast(bf16x8, v);
    }
  }
  // the wave's first and last query: tiles past the last are left out, tiles up to the first need no mask
  const int wq0 = qstart + min(tile * QT + wid * RB * 16 / G, qlen - 1);
  const int wq1 = qstart + min(tile * QT + (wid * RB * 16 + 16 * RB - 1) / G, qlen - 1);

  f32x4 o[RB][D / 16];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int n = 0; n < D / 16; ++n) o[b][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run[RB], l_run[RB];   // row li's maximum so far, log2; this lane's share of its sum
#pragma unroll
  for (int b = 0; b < RB; ++b) m_run[b] = -INFINITY, l_run[b] = 0.f;

  f32x4 sacc[RB][KT / 16];
  bf16x8 pa[RB][KT / 32];
  // S^T = K . Q^T for 4 key sub-tiles of 16; lane (li, g) reads key row 16m + li, d 32kk + 8g
  auto scores = [&](const char* kl) {
#pragma unroll
    for (int m = 0; m < KT / 16; ++m) {
      const int kr = 16 * m + li;
#pragma unroll
      for (int b = 0; b < RB; ++b) sacc[b][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < D / 32; ++kk) {
        const bf16x8 ka = *reinterpret_cast<const bf16x8*>(kl + kr * (D * 2) + 16 * ((4 * kk + g) ^ (kr & 15)));
#pragma unroll
        for (int b = 0; b < RB; ++b) sacc[b][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[b][kk], sacc[b][m], 0, 0, 0);
      }
    }
  };
  // lane holds S[row li][key kbase + 16m + 4g + i]
  auto weights = [&](int kbase) {
    if (kbase + KT - 1 > wq0) {
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int m = 0; m < KT / 16; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kbase + m * 16 + g * 4 + i > qpos[b]) sacc[b][m][i] = -INFINITY;
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      // the scores against the maximum so far: only if one of the rows has outgrown it do the lanes meet for the new one
      const float base = m_run[b] == -INFINITY ? 0.f : m_run[b];
      float top[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
      for (int m = 0; m < KT / 16; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sacc[b][m][i] = fmaf(sacc[b][m][i], scale, -base);
          top[i] = fmaxf(top[i], sacc[b][m][i]);
        }
      float over = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
      if (__any(over > 0.f || m_run[b] == -INFINITY)) {
        over = row_max(over);
        const float m_new = fmaxf(m_run[b], base + over);
        const float alpha = m_run[b] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[b] - m_new);
        const float d = m_new == -INFINITY ? 0.f : m_new - base;
        l_run[b] *= alpha;
        m_run[b] = m_new;
#pragma unroll
        for (int m = 0; m < KT / 16; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) sacc[b][m][i] -= d;
#pragma unroll
        for (int n = 0; n < D / 16; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[b][n][i] *= alpha;
      }
      // P as B operand: k-step st covers keys 32st..32st+31 in the permuted order
      // slot j<4 -> key 32st + 4g + j ; slot j>=4 -> key 32st + 16 + 4g + (j-4)
      f32x4 rs = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < KT / 16; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float w = __builtin_amdgcn_exp2f(sacc[b][m][i]);
          rs[i] += w;
          pa[b][m >> 1][4 * (m & 1) + i] = (__bf16)w;
        }
      l_run[b] += (rs[0] + rs[1]) + (rs[2] + rs[3]);
    }
  };
  auto values = [&](const char* vl) {
    const int qd = li >> 2, pd = li & 3;  // tr-read lane roles: row q, column group p
#pragma unroll
    for (int st = 0; st < KT / 32; ++st) {
      const int r0 = 32 * st + 4 * g + qd;
      const int r1 = r0 + 16;
#pragma unroll
      for (int n = 0; n < D / 16; ++n) {
        const int col = 16 * n + 4 * pd;
        const int ch = col >> 3, hb = (col & 7) * 2;
        const lds_bf16x4* a0 = (const lds_bf16x4*)(vl + r0 * (D * 2) + 16 * (ch ^ v_swz(r0)) + hb);
        const lds_bf16x4* a1 = (const lds_bf16x4*)(vl + r1 * (D * 2) + 16 * (ch ^ v_swz(r1)) + hb);
        const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)a0);
        const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)a1);
        bf16x8 vb;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vb[j] = v0[j]; vb[4 + j] = v1[j]; }
#pragma unroll
        for (int b = 0; b < RB; ++b) o[b][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, pa[b][st], o[b][n], 0, 0, 0);
      }
    }
  };
  fetch_v();
  ids();
  stage_k(0);
  mask_v(0);
  stage_v(0);
  auto ahead = [&](int t) {
    if (t >= ntiles) return;
    fetch_k();
    keep();
    fetch_v();
    ids();
  };
  ahead(1);
  lds_barrier();
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) {
      stage_k((t + 1) & 1);          // (tile t - 1 was read before the last barrier)
      mask_v(t + 1);
      stage_v((t + 1) & 1);
      ahead(t + 2);
    }
    const int kbase = t * ST + share * KT;
    if (kbase <= wq1) {
      scores(klds[t & 1] + share * (KT * D * 2));
      weights(kbase);
      values(vlds[t & 1] + share * (KT * D * 2));
    }
    lds_barrier();                   // tile t has been read and tile t + 1 written
  }

  float l_row[RB];                   // row li's sum
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    l_row[b] = row_sum(l_run[b]);
  }
  if constexpr (KS == 2) {           // the second share's sums join the first one's, through the staged K
    static_assert(RW * RB * (D / 16) * 64 * 16 <= 2 * ST * D * 2, "room for a share's sums");
    if (share == 1 && kv_end <= KT) return;
    f32x4* os = reinterpret_cast<f32x4*>(klds[0]);
    float* ms = reinterpret_cast<float*>(vlds[0]);
    if (share == 1) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
#pragma unroll
        for (int n = 0; n < D / 16; ++n) os[((wid * RB + b) * (D / 16) + n) * 64 + lane] = o[b][n];
        if (g == 0) {
          ms[((wid * RB + b) * 16 + li) * 2] = m_run[b];
          ms[((wid * RB + b) * 16 + li) * 2 + 1] = l_row[b];
        }
      }
    }
    if (kv_end > KT) lds_barrier();
    if (share == 1) return;
#pragma unroll
    for (int b = 0; b < RB && kv_end > KT; ++b) {
      const float m1 = ms[((wid * RB + b) * 16 + li) * 2], l1 = ms[((wid * RB + b) * 16 + li) * 2 + 1];
      const float m = fmaxf(m_run[b], m1);
      const float a0 = m_run[b] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[b] - m);
      const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - m);
      l_row[b] = l_row[b] * a0 + l1 * a1;
#pragma unroll
      for (int n = 0; n < D / 16; ++n) {
        const f32x4 o1 = os[((wid * RB + b) * (D / 16) + n) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[b][n][i] = o[b][n][i] * a0 + o1[i] * a1;
      }
    }
  }

  // ---- normalise and store: o[b][n][i] = O[row li][d 16n + 4g + i]
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const float inv_l = l_row[b] > 0.f ? 1.f / l_row[b] : l_row[b] == 0.f ? 0.f : l_row[b];   // (NaN stays one)
    const int orow = (wid * RB + b) * 16 + li;
    const int r = tile * QT + orow / G, oh = kvh * G + orow % G;
    if (r < qlen) {
      bf16_t* op = out + ((size_t)(q0 + r) * nq + oh) * D + 4 * g;
#pragma unroll
      for (int n = 0; n < D / 16; ++n)
        stf4(op + 16 * n, f32x4{o[b][n][0] * inv_l, o[b][n][1] * inv_l, o[b][n][2] * inv_l, o[b][n][3] * inv_l});
    }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

K8S_CHECK_UNIT(attn_prefill)

// form 4: 64 rows a workgroup; 5: 64, the keys shared by two halves of 8 waves; 8: 128, shared; 16: 256 (which when: ops/__init__.py _prefill_form)
extern "C" int k8s_paged_prefill_attention(void* out, const void* q, const void* k_cache, const void* v_cache,
                                           const int* cu_q, const int* context_lens, const int* block_tables,
                                           float scale, int num_seqs, int max_qlen, int nq, int nkv, int D,
                                           int block_size, int max_blocks, int form, hipStream_t stream) {
  if (num_seqs <= 0 || max_qlen <= 0) return 0;
  if (D != 128 || nq % nkv != 0 || (uintptr_t)out % 8 || (form != 4 && form != 5 && form != 8 && form != 16)) return -1;
  const int G = nq / nkv;
  const float sl2 = scale * 1.4426950408889634f;
#define PF(GG, RB, NW, KS)                                                                                   \
  {                                                                                                          \
    constexpr int QT = 16 * RB * NW / KS / GG;                                                               \
    const int tiles = (max_qlen + QT - 1) / QT;                                                              \
    paged_prefill_kernel<GG, RB, NW, KS><<<dim3(tiles * nkv, 1, num_seqs), 64 * NW, 0, stream>>>(            \
        (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu_q, context_lens,  \
        block_tables, sl2, nq, nkv, block_size, max_blocks, tiles);                                          \
  }
#define PFR(GG) \
  if (form == 16) PF(GG, 2, 8, 1) else if (form == 8) PF(GG, 2, 8, 2) else if (form == 4) PF(GG, 1, 4, 1) else PF(GG, 1, 8, 2)
  switch (G) {  // query heads per kv head (Llama-3.3-70B: 8; Llama-3-8B: 4)
    case 1: PFR(1) break;
    case 2: PFR(2) break;
    case 4: PFR(4) break;
    case 8: PFR(8) break;
    case 16: PFR(16) break;
    default: return -1;
  }
#undef PFR
#undef PF
  return (int)hipGetLastError();
}
