// Linear attention under a constant decay per head on the matrix cores (long bf16 portions):
//   q = silu(zq), k = silu(zk), v = silu(zv);  S_t = a S_(t-1) + k_t v_t^T;  o_t = S_t^T q_t
// (the recurrence of gated_scan.hip's KIND 3; that kernel runs decoding, short portions, fp32 and other sizes).
// A portion is cut into chunks of 64 tokens.  With i, j counting from the chunk's first token and S0 the state before it,
//   o_i = a^(i + 1) S0^T q_i + sum_(j <= i) a^(i - j) (q_i . k_j) v_j
//   S0' = a^n S0 + sum_j a^(n - 1 - j) k_j v_j^T                            (n: the chunk's tokens)
// so everything but the walk over the chunks is a product of tiles.  Three kernels:
//   decay_chunk_kernel   per (chunk, head, slice of value columns): the chunk's own sum of k v^T, fp32;
//   decay_prefix_kernel  per (sequence, head, state elements): walks the sequence's chunks from the slot's state, leaves
//                        every chunk's S0 in the place of its sum and, at the end, the slot's new state;
//   decay_out_kernel     per (chunk, head, slice of value columns): the outputs, fp32.
// Where no portion is longer than one chunk, or two of them and there are more than 16 workgroups, the last does it all.
// Exactness: q, k, v enter the products as bf16 (activations); the decay weights, the scores and the state are fp32 and
// enter a product as two bf16 terms (hi + lo, 16 bits of mantissa together); sums are fp32.
//
// Fragments of v_mfma_f32_16x16x32_bf16 here: lane (li = lane & 15, g = lane >> 4); operand A holds row li, operand B
// column li, at the eight k indices 4 g + j (slot j < 4) and 16 + 4 g + (j - 4) (slot j >= 4) -- the same order in both,
// which is what the transposing LDS read and the accumulator layout (row 4 g + i, column li) give without a shuffle.
#include "common.h"

namespace k8sllm {

typedef __attribute__((address_space(3))) bf16x4 ds_bf16x4;

constexpr int DSC_L = 64;          // tokens per chunk
constexpr int DSC_VS = 128;        // value columns per workgroup
constexpr int DSC_PAD = 8;         // LDS row padding, elements

struct DecayArgs {
  const bf16_t* proj;
  long ld;
  int cq, ck, cv;                  // column offsets of q, k, v
  const float* decay;              // [H]
  const int* cu_q;
  const int* seq_slots;
  const int* positions;
  int nseq, H, D, V, R;            // R heads share a group's q and k
};

__device__ __forceinline__ float fast_silu(float z) { return z * __builtin_amdgcn_rcpf(1.f + __expf(-z)); }

// 8 bf16 -> silu -> 8 floats
__device__ __forceinline__ void silu8(u32x4 u, float* y) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    y[2 * i] = fast_silu(lo_bf(u[i]));
    y[2 * i + 1] = fast_silu(hi_bf(u[i]));
  }
}
__device__ __forceinline__ u32x4 pack8(const float* y) {
  return u32x4{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]), pack_bf2(y[4], y[5]), pack_bf2(y[6], y[7])};
}
__device__ __forceinline__ bf16x8 join4(bf16x4 a, bf16x4 b) {
  bf16x8 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) { r[j] = a[j]; r[4 + j] = b[j]; }
  return r;
}
// fragment of LDS rows read along the row: row `r`, k indices k0 + 4 g + .., k0 + 16 + 4 g + ..
__device__ __forceinline__ bf16x8 row_frag(const bf16_t* base, int stride, int r, int k0, int g) {
  const bf16_t* p = base + r * stride + k0 + 4 * g;
  return join4(*reinterpret_cast<const bf16x4*>(p), *reinterpret_cast<const bf16x4*>(p + 16));
}
// fragment across LDS rows: column c0 + li, k indices are the rows k0 + 4 g + .., k0 + 16 + 4 g + ..
__device__ __forceinline__ bf16x8 col_frag(bf16_t* base, int stride, int c0, int k0, int li, int g) {
  bf16_t* p = base + (k0 + 4 * g + (li >> 2)) * stride + c0 + 4 * (li & 3);
  return join4(__builtin_amdgcn_ds_read_tr16_b64_v4bf16((ds_bf16x4*)p),
               __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ds_bf16x4*)(p + 16 * stride)));
}
// Keeps the compiler from holding every LDS and row address of a loop's body in registers across its rounds (hundreds, spilled)
__device__ __forceinline__ void own_addresses(int& tid, int& li, int& g) { asm volatile("" : "+v"(tid), "+v"(li), "+v"(g)); }
// 64 rows of N 16-byte pieces (the chunk's tokens, from `p`, columns up to `width`) on their way into registers; rows past the
// chunk's `n` repeat its last one (their weights are zero), columns outside are zeros, which silu leaves
template <int NTHR, int N, int PER>
__device__ __forceinline__ void load_rows(u32x4 (&z)[PER], int tid, const bf16_t* p, long ld, int n, int width) {
  static_assert(PER * NTHR >= DSC_L * N, "all of the rows");
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int idx = tid + NTHR * i, r = min(idx / N, n - 1), c = (idx % N) * 8;
    z[i] = u32x4{0u, 0u, 0u, 0u};
    if (c < width) z[i] = *reinterpret_cast<const u32x4*>(p + (size_t)r * ld + c);
  }
}
// ... silu, bf16, to LDS rows; pieces from column `cols` on are left out
template <int NTHR, int N, int PER>
__device__ __forceinline__ void store_rows(int tid, bf16_t* dst, int stride, const u32x4 (&z)[PER], int cols) {
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int idx = tid + NTHR * i, r = idx / N, c = (idx % N) * 8;
    float y[8];
    silu8(z[i], y);
    if ((DSC_L * N % NTHR == 0 || r < DSC_L) && c < cols) *reinterpret_cast<u32x4*>(dst + r * stride + c) = pack8(y);
  }
}
// ... times decay^(n - 1 - row) of the table pw, as two bf16 terms
template <int NTHR, int N, int PER>
__device__ __forceinline__ void store_faded(int tid, bf16_t* hi, bf16_t* lo, int stride, const u32x4 (&z)[PER], const float* pw, int n) {
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int idx = tid + NTHR * i, r = idx / N, c = (idx % N) * 8;
    if (DSC_L * N % NTHR != 0 && r >= DSC_L) continue;
    float y[8], h8[8], l8[8];
    silu8(z[i], y);
    const float w = r < n ? pw[n - 1 - r] : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = bf_round(y[e]) * w;
      h8[e] = bf_round(f);
      l8[e] = f - h8[e];
    }
    *reinterpret_cast<u32x4*>(hi + r * stride + c) = pack8(h8);
    *reinterpret_cast<u32x4*>(lo + r * stride + c) = pack8(l8);
  }
}

// acc += sum over the chunk's tokens of k v^T, keys as two terms: value columns 16 nt .., all key channels
template <int KK>
__device__ __forceinline__ void add_chunk(f32x4 (&acc)[2 * KK], bf16_t* khi, bf16_t* klo, bf16_t* vl, int LDV, int nt, int n, int li, int g) {
  constexpr int LDK = 32 * KK + DSC_PAD;
#pragma unroll
  for (int k0 = 0; k0 < DSC_L; k0 += 32) {
    if (k0 >= n) break;
    const bf16x8 vf = col_frag(vl, LDV, 16 * nt, k0, li, g);
#pragma unroll
    for (int d = 0; d < 2 * KK; ++d) {
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(col_frag(klo, LDK, 16 * d, k0, li, g), vf, acc[d], 0, 0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(col_frag(khi, LDK, 16 * d, k0, li, g), vf, acc[d], 0, 0, 0);
    }
  }
}

// A chunk's / state's record: tile (nt, dt) of 16 key channels x 16 value columns in accumulator order, element
// ((nt DT + dt) 64 + lane) 4 + i = S[16 dt + 4 g + i][16 nt + li], DT = 2 KK tiles of key channels (zero-padded).
template <int KK, int NTHR>
__global__ __launch_bounds__(NTHR) void decay_chunk_kernel(float* __restrict__ rec, DecayArgs A) {
  constexpr int DT = 2 * KK, DP = 32 * KK, LDK = DP + DSC_PAD, PER = (4 * KK * DSC_L + NTHR - 1) / NTHR;
  extern __shared__ __attribute__((aligned(16))) char smem_d[];
  __shared__ float pw[DSC_L];
  const WkvChunk ck = wkv_find_chunk(blockIdx.x, A.cu_q, A.positions, A.nseq, DSC_L);
  if (ck.s < 0) return;
  const int hd = blockIdx.y, v0 = blockIdx.z * DSC_VS;
  const int a0 = A.cu_q[ck.s] + ck.c * DSC_L, n = min(DSC_L, A.cu_q[ck.s + 1] - a0);
  const int vw = min(DSC_VS, A.V - v0), NT = (vw + 15) / 16, LDV = 16 * NT + DSC_PAD;
  bf16_t* khi = reinterpret_cast<bf16_t*>(smem_d);       // [64][LDK]
  bf16_t* klo = khi + DSC_L * LDK;
  bf16_t* vl = klo + DSC_L * LDK;                        // [64][LDV]
  const int tid = threadIdx.x;
  u32x4 zk[PER], zv[16 * DSC_L / NTHR];
  const bf16_t* row = A.proj + (size_t)a0 * A.ld;
  load_rows<NTHR, 4 * KK>(zk, tid, row + A.ck + (long)(hd / A.R) * A.D, A.ld, n, A.D);
  load_rows<NTHR, 16>(zv, tid, row + A.cv + (long)hd * A.V + v0, A.ld, n, vw);
  if (tid < DSC_L) pw[tid] = powf(A.decay[hd], (float)tid);
  __syncthreads();
  store_faded<NTHR, 4 * KK>(tid, khi, klo, LDK, zk, pw, n);
  store_rows<NTHR, 16>(tid, vl, LDV, zv, 16 * NT);
  __syncthreads();
  const int lane = tid & 63, wave = tid >> 6, li = lane & 15, g = lane >> 4, ntt = (A.V + 15) / 16;
  if (wave >= NT) return;
  f32x4 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  add_chunk<KK>(acc, khi, klo, vl, LDV, wave, n, li, g);
  float* r = rec + ((size_t)blockIdx.x * A.H + hd) * ((size_t)ntt * DT * 256) + ((size_t)(v0 / 16 + wave) * DT * 64 + lane) * 4;
#pragma unroll
  for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(r + d * 256) = acc[d];
}

// Thread: the four elements of one lane of one tile.  A chunk's record is replaced by the state before it.
__global__ __launch_bounds__(256) void decay_prefix_kernel(float* __restrict__ rec, float* __restrict__ state, DecayArgs A, int KK) {
  const int s = blockIdx.x, hd = blockIdx.y;
  int first = 0;
  for (int y = 0; y < s; ++y) {
    const int a = A.cu_q[y], len = A.cu_q[y + 1] - a;
    first += (len > 0 && A.positions[a] >= 0) ? (len + DSC_L - 1) / DSC_L : 0;
  }
  const int a = A.cu_q[s], len = A.cu_q[s + 1] - a;
  if (len <= 0 || A.positions[a] < 0) return;
  const int nch = (len + DSC_L - 1) / DSC_L;
  const int DT = 2 * KK, ntt = (A.V + 15) / 16, nvec = ntt * DT * 64;
  const int e = blockIdx.z * blockDim.x + threadIdx.x;
  if (e >= nvec) return;
  const int lane = e & 63, tile = e >> 6, nt = tile / DT, dt = tile - nt * DT;
  const int v = 16 * nt + (lane & 15), d0 = 16 * dt + 4 * (lane >> 4);
  const size_t recf = (size_t)nvec * 4;                  // floats of a record
  float* st = state + ((size_t)A.seq_slots[s] * A.H + hd) * ((size_t)A.D * A.V);
  const bool zero = A.positions[a] == 0;
  float* p = rec + ((size_t)first * A.H + hd) * recf + (size_t)e * 4;
  const size_t step = (size_t)A.H * recf;
  constexpr int PF = 8;                                  // records in flight
  f32x4 buf[PF], X = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < PF; ++i)
    if (i < nch) buf[i] = *reinterpret_cast<const f32x4*>(p + i * step);
  const bool live = d0 < A.D && v < A.V;                 // (D is a multiple of 8)
  if (!zero && live) {
#pragma unroll
    for (int i = 0; i < 4; ++i) X[i] = st[(unsigned)((d0 + i) * A.V + v)];
  }
  const float dec = A.decay[hd], full = powf(dec, (float)DSC_L), last = powf(dec, (float)(len - (nch - 1) * DSC_L));
  for (int c0 = 0; c0 < nch; c0 += PF) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int c = c0 + i;
      if (c < nch) {
        const f32x4 U = buf[i];
        if (c + PF < nch) buf[i] = *reinterpret_cast<const f32x4*>(p + (c + PF) * step);
        if (c > 0 || !zero) *reinterpret_cast<f32x4*>(p + c * step) = X;
        const float w = c + 1 < nch ? full : last;
#pragma unroll
        for (int j = 0; j < 4; ++j) X[j] = fmaf(w, X[j], U[j]);
      }
    }
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < 4; ++i) st[(unsigned)((d0 + i) * A.V + v)] = X[i];
  }
}

// Waves: first the scores of 16 queries each (of 8 waves two share them) against the keys up to them, weighted, into LDS; then
// each its 16 value columns for all 64 queries.  ONCE: workgroups (sequence, head, slice of value columns) walk a short
// portion's chunks, the state in registers from its slot and back: one launch instead of three.
// A few hundred workgroups of short work: bound by what a wave executes one after the other (loads, silu and its exponentials,
// addresses), not by memory or the matrix cores.  Hence 8 waves of 16 value columns (4 of 32 before), every load under way
// before the first use, powers by a table, the queries staged beside the keys, states handed on as one fp32 record.  All three
// kernels, 128 channels, before and after, us: 2048 tokens of 16 heads 61.6 -> 50, of 32 96.4 -> 79; 512 of 32 41.7 -> 34;
// 100 of 16 26.0 -> 19.5; 60 of 16 24.9 -> 11.6.  ONCE takes 12 us and 8 for a second chunk, the three kernels 19 and more with every
// workgroup, us, three / ONCE: 128 tokens of 16 heads 20.4 / 20.4, of 8 19.3 / 20.3, of 32 23.3 / 20.8, 3 x 128 of 4 (2 slices) 19.8 / 19.4,
// 4 x 100 of 32 40 / 22, 16 x 128 of 32 109 / 51.  Segments of two chunks a workgroup (half the records) were slower below a
// thousand workgroups: 2048 tokens of 16 heads 54.9 against 50.1.
template <int KK, int NTHR, bool ONCE>
__global__ __launch_bounds__(NTHR, ONCE ? 1 : NTHR / 128) void decay_out_kernel(float* __restrict__ out, const float* __restrict__ rec, float* __restrict__ state,
                                                           DecayArgs A) {
  constexpr int DT = 2 * KK, DP = 32 * KK, LDK = DP + DSC_PAD, LDP = DSC_L + DSC_PAD, PER = (4 * KK * DSC_L + NTHR - 1) / NTHR;
  extern __shared__ __attribute__((aligned(16))) char smem_d[];
  __shared__ float pw[DSC_L + 1];
  const int hd = blockIdx.y, v0 = blockIdx.z * DSC_VS;
  WkvChunk ck{(int)blockIdx.x, 0, 1};
  if constexpr (!ONCE) ck = wkv_find_chunk(blockIdx.x, A.cu_q, A.positions, A.nseq, DSC_L);
  if (ck.s < 0) return;
  int a0 = A.cu_q[ck.s] + (ONCE ? 0 : ck.c * DSC_L);
  const int end = ONCE ? A.cu_q[ck.s + 1] : min(a0 + DSC_L, A.cu_q[ck.s + 1]);
  if (ONCE && a0 >= end) return;
  const int p0 = A.positions[a0];
  if (ONCE && p0 < 0) return;
  bool none = p0 == 0;                                   // nothing before this chunk
  const int NT = (min(DSC_VS, A.V - v0) + 15) / 16, LDV = 16 * NT + DSC_PAD, ntt = (A.V + 15) / 16;
  bf16_t* kl = reinterpret_cast<bf16_t*>(smem_d);        // [64][LDK]
  bf16_t* ql = kl + DSC_L * LDK;                         // [64][LDK]
  bf16_t* ph = ql + DSC_L * LDK;                         // [64][LDP]
  bf16_t* pl = ph + DSC_L * LDP;
  bf16_t* vl = pl + DSC_L * LDP;                         // [64][LDV]
  int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  int li = lane & 15, g = lane >> 4;
  const bool mine = wave < NT;                           // 16 value columns a wave
  const int nt = mine ? wave : 0, rw = wave & 3, half = wave >> 2;   // rw: the 16 rows whose scores it takes part in
  const int sv = v0 + 16 * nt + li;
  const bool live = mine && sv < A.V;
  // every load under way before any is used
  const bf16_t* kp = A.proj + A.ck + (long)(hd / A.R) * A.D;
  const bf16_t* qp = A.proj + A.cq + (long)(hd / A.R) * A.D;
  const bf16_t* vp = A.proj + A.cv + (long)hd * A.V + v0;
  const int vw = min(DSC_VS, A.V - v0);
  u32x4 zk[PER], zq[PER], zv[16 * DSC_L / NTHR];
  int n = min(DSC_L, end - a0);
  load_rows<NTHR, 4 * KK>(zk, tid, kp + (size_t)a0 * A.ld, A.ld, n, A.D);
  load_rows<NTHR, 4 * KK>(zq, tid, qp + (size_t)a0 * A.ld, A.ld, n, A.D);
  load_rows<NTHR, 16>(zv, tid, vp + (size_t)a0 * A.ld, A.ld, n, vw);
  f32x4 X[DT];                                           // the state, tiles in accumulator order
#pragma unroll
  for (int d = 0; d < DT; ++d) X[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float* st = nullptr;
  if constexpr (ONCE) {
    st = state + ((size_t)A.seq_slots[ck.s] * A.H + hd) * ((size_t)A.D * A.V);
    if (!none && live) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
        if (16 * d + 4 * g < A.D) {                      // (D is a multiple of 8)
#pragma unroll
          for (int i = 0; i < 4; ++i) X[d][i] = st[(unsigned)((16 * d + 4 * g + i) * A.V + sv)];
        }
    }
  } else if (!none) {
    const float* r = rec + ((size_t)blockIdx.x * A.H + hd) * ((size_t)ntt * DT * 256);
    const unsigned o = ((unsigned)((v0 / 16 + nt) * DT) * 64 + lane) * 4;
#pragma unroll
    for (int d = 0; d < DT; ++d) X[d] = *reinterpret_cast<const f32x4*>(r + (o + d * 256));
  }
  if (threadIdx.x <= DSC_L) pw[threadIdx.x] = powf(A.decay[hd], (float)threadIdx.x);
  for (;;) {
    own_addresses(tid, li, g);
    store_rows<NTHR, 4 * KK>(tid, kl, LDK, zk, DP);
    store_rows<NTHR, 4 * KK>(tid, ql, LDK, zq, DP);
    store_rows<NTHR, 16>(tid, vl, LDV, zv, 16 * NT);
    __syncthreads();
    if (16 * rw < n) {
      bf16x8 qf[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) qf[kk] = row_frag(ql, LDK, 16 * rw + li, 32 * kk, g);
      // key tiles up to the rows' own and the one that shares its 32 keys; of 8 waves every other one
      for (int jt = half; jt <= (rw | 1); jt += NTHR / 256) {
        f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
        if (jt <= rw) {
#pragma unroll
          for (int kk = 0; kk < KK; ++kk)
            sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(row_frag(kl, LDK, 16 * jt + li, 32 * kk, g), qf[kk], sc, 0, 0, 0);
        }
        // sc[i]: key 16 jt + 4 g + i, query 16 rw + li
        float h[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int age = 16 * rw + li - (16 * jt + 4 * g + i);
          const float p = age >= 0 ? sc[i] * pw[age] : 0.f;
          h[i] = bf_round(p);
          l[i] = p - h[i];
        }
        const int o = (16 * rw + li) * LDP + 16 * jt + 4 * g;
        *reinterpret_cast<uint2*>(ph + o) = make_uint2(pack_bf2(h[0], h[1]), pack_bf2(h[2], h[3]));
        *reinterpret_cast<uint2*>(pl + o) = make_uint2(pack_bf2(l[0], l[1]), pack_bf2(l[2], l[3]));
      }
    }
    __syncthreads();
    f32x4 acc[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!none) {
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        bf16x8 sh, sl;                                   // two terms, B fragments (slot j: tile 2 kk + j / 4)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float f = X[2 * kk + (e >> 2)][e & 3], h = bf_round(f);
          sh[e] = (__bf16)h;
          sl[e] = (__bf16)(f - h);
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          const bf16x8 a = row_frag(ql, LDK, 16 * rt + li, 32 * kk, g);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, sl, acc[rt], 0, 0, 0);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, sh, acc[rt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][i] *= pw[16 * rt + 4 * g + i + 1];
    }
#pragma unroll
    for (int k0 = 0; k0 < DSC_L; k0 += 32) {
      if (k0 >= n) break;
      const bf16x8 vf = col_frag(vl, LDV, 16 * nt, k0, li, g);
#pragma unroll
      for (int rt = k0 / 16; rt < 4; ++rt) {
        if (16 * rt >= n) break;                         // those rows' scores were not written
        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(row_frag(pl, LDP, 16 * rt + li, k0, g), vf, acc[rt], 0, 0, 0);
        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(row_frag(ph, LDP, 16 * rt + li, k0, g), vf, acc[rt], 0, 0, 0);
      }
    }
    if (live) {
      const int ldo = A.H * A.V;
      float* op = out + (size_t)a0 * ldo + (size_t)hd * A.V;
      const unsigned o = (unsigned)(4 * g * ldo + sv);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        if (16 * rt + 16 <= n) {
#pragma unroll
          for (int i = 0; i < 4; ++i) op[o + (unsigned)((16 * rt + i) * ldo)] = acc[rt][i];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * rt + 4 * g + i < n) op[o + (unsigned)((16 * rt + i) * ldo)] = acc[rt][i];
        }
      }
    }
    if constexpr (!ONCE) {
      break;
    } else {
      const int m = n;
      a0 += DSC_L;
      n = min(DSC_L, end - a0);
      __syncthreads();                                     // keys and scores have been read: the faded keys take their place
      static_assert(LDK <= 2 * LDP, "the faded keys' second term in the scores' place");
      store_faded<NTHR, 4 * KK>(tid, kl, ph, LDK, zk, pw, m);
      if (n > 0) {                                         // the next chunk's rows on their way
        load_rows<NTHR, 4 * KK>(zk, tid, kp + (size_t)a0 * A.ld, A.ld, n, A.D);
        load_rows<NTHR, 4 * KK>(zq, tid, qp + (size_t)a0 * A.ld, A.ld, n, A.D);
        load_rows<NTHR, 16>(zv, tid, vp + (size_t)a0 * A.ld, A.ld, n, vw);
      }
      __syncthreads();
      const float w = pw[m];
#pragma unroll
      for (int d = 0; d < DT; ++d) X[d] *= w;
      add_chunk<KK>(X, kl, ph, vl, LDV, nt, m, li, g);
      none = false;
      if (n <= 0) break;
      __syncthreads();                                     // they go where these were read
      }
  }
  if constexpr (ONCE) {
    if (live) {
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        if (16 * d + 4 * g >= A.D) break;
#pragma unroll
        for (int i = 0; i < 4; ++i) st[(unsigned)((16 * d + 4 * g + i) * A.V + sv)] = X[d][i];
      }
    }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

// Whether these sizes run here (else k8s_gated_scan): rows of 16 bytes, at most 128 key channels.
extern "C" int k8s_decay_scan_ok(int D, int V) { return D > 0 && D <= 128 && D % 8 == 0 && V > 0 && V <= 256 && V % 8 == 0; }

// Bytes of workspace: per chunk and head one fp32 record.
extern "C" long long k8s_decay_scan_workspace(int T, int nseq, int H, int D, int V) {
  const long long chunks = (T + DSC_L - 1) / DSC_L + nseq;
  const long long rec = (long long)((V + 15) / 16) * 2 * ((D + 31) / 32) * 256;
  return chunks * H * rec * 4;
}

// Whether portions of at most max_qlen tokens run in one launch, which needs no workspace (figures at decay_out_kernel).
extern "C" int k8s_decay_scan_once(int nseq, int H, int V, int max_qlen) {
  return max_qlen > 0 && (max_qlen <= DSC_L || (max_qlen <= 2 * DSC_L && (long long)nseq * H * ((V + DSC_VS - 1) / DSC_VS) > 16));
}

// proj bf16 [T, ld] (16-byte aligned rows and parts); out fp32 [T, H V]; state [slots, H, D V] fp32, updated in place.  max_qlen: no portion
// is longer.
extern "C" int k8s_decay_scan(float* out, const void* proj, long ld, int cq, int ck, int cv, const float* decay,
                              float* state, const int* cu_q, const int* seq_slots, const int* positions, int nseq, int H,
                              int D, int V, int R, int T, int max_qlen, void* ws, hipStream_t s) {
  if (T <= 0 || nseq <= 0) return 0;
  const bool once = k8s_decay_scan_once(nseq, H, V, max_qlen) != 0;
  if (!k8s_decay_scan_ok(D, V) || H <= 0 || H > 65535 || R <= 0 || H % R || (ws == nullptr && !once) || decay == nullptr) return -1;
  if (ld % 8 || cq % 8 || ck % 8 || cv % 8 || ((uintptr_t)proj & 15)) return -1;
  const DecayArgs A{(const bf16_t*)proj, ld, cq, ck, cv, decay, cu_q, seq_slots, positions, nseq, H, D, V, R};
  const int KK = (D + 31) / 32, slices = (V + DSC_VS - 1) / DSC_VS, ntt = (V + 15) / 16;
  const int chunks = (T + DSC_L - 1) / DSC_L + nseq;
  const size_t recf = (size_t)ntt * 2 * KK * 256;
  float* rec = (float*)ws;
  const int nt = ntt < 8 ? ntt : 8, LDK = 32 * KK + DSC_PAD, LDV = 16 * nt + DSC_PAD;
  const size_t lds1 = (size_t)DSC_L * (2 * LDK + LDV) * 2;
  const size_t lds3 = (size_t)DSC_L * (2 * LDK + 2 * (DSC_L + DSC_PAD) + LDV) * 2;
  const dim3 grid(chunks, H, slices), pgrid(nseq, H, (unsigned)((recf / 4 + 255) / 256));
#define K8S_DS(KK_, NTHR)                                                             \
  do {                                                                                \
    static bool grown = false;   /* more LDS than a launch gets by default */         \
    if (!grown) {                                                                     \
      constexpr int most = DSC_L * (2 * (32 * KK_ + DSC_PAD) + 2 * (DSC_L + DSC_PAD) + DSC_VS + DSC_PAD) * 2; \
      for (const void* k : {(const void*)decay_out_kernel<KK_, NTHR, true>, (const void*)decay_out_kernel<KK_, NTHR, false>}) { \
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, most); \
        if (e != hipSuccess) return (int)e;                                           \
      }                                                                               \
      grown = true;                                                                   \
    }                                                                                 \
    if (once) {                                                                       \
      decay_out_kernel<KK_, NTHR, true><<<dim3(nseq, H, slices), NTHR, lds3, s>>>(out, nullptr, state, A); \
      break;                                                                          \
    }                                                                                 \
    decay_chunk_kernel<KK_, NTHR><<<grid, NTHR, lds1, s>>>(rec, A);                   \
    decay_prefix_kernel<<<pgrid, 256, 0, s>>>(rec, state, A, KK);              \
    decay_out_kernel<KK_, NTHR, false><<<grid, NTHR, lds3, s>>>(out, rec, nullptr, A); \
  } while (0)
#define K8S_DS_N(KK_)                 \
  do {                                \
    if (nt <= 4) K8S_DS(KK_, 256);    \
    else K8S_DS(KK_, 512);            \
  } while (0)
  if (KK == 1) K8S_DS_N(1);
  else if (KK == 2) K8S_DS_N(2);
  else if (KK == 3) K8S_DS_N(3);
  else K8S_DS_N(4);
#undef K8S_DS_N
#undef K8S_DS
  return (int)hipGetLastError();
}
