// fp32 products of many tiles: C[M, N] = A[M, K] W[N, K]^T on v_mfma_f32_16x16x4_f32 (fp32 products and sums), K % 32 == 0.
// They take what gemm_f32_parts.hip's rule leaves them: bf16 outputs, and sizes at which they are within a tenth of its tiles.
//
// A workgroup of 4 waves owns 64 columns x 16 FQ rows (swapped orientation C^T = W A^T; a wave 16 columns x all rows), so the
// row count is padded to 16 and FQ is chosen for the tiles to fill the CUs' last round.  k in 32-deep stages of 128-byte rows
// through a ring of NS LDS slots filled by LDS-DMA (XOR swizzle on the source: conflict-free 16-byte fragment reads), one
// barrier a stage; the fragments of the next 16 k are read between the products of the current ones.
// Every 32, 64 (K >= 1024) or 128 (K >= 2048) k the products' registers are added to a second set: chains of that many terms
// and then of their number, whatever the tile.  Error against 64 bits, 2-norm: K = 2048 2.2e-7, 8192 2.5e-7 (2.9e-7 and 5.8e-7
// with the eight shares of gemm_f32_kernel).
//
// Bound by the matrix rate (157 TFLOP/s at 2.4 GHz; the clock holds 2.25 here): 85 % of a busy CU's cycles with two workgroups
// on it, 70 - 80 % with one (a stage's barrier and waits cost about 350 cycles; a ring of 8 slots changes nothing).  us with the
// launch: 333 x 16384 x 2048 258 -> 175 (three rounds of 112-row tiles), 200 x 16384 x 2048 165 -> 116.
#include <type_traits>

#include "common.h"

namespace k8sllm {

template <int N>
__device__ __forceinline__ void f32_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

struct F32Args {
  void* C;
  const float *A, *W;
  int M, N, K, mt, nt, batch;       // mt row tiles; listed tiles: PER blocks for each
  long lda, ldw, ldc, sA, sW, sC;
  const int *a_rows, *tiles;
  int vec;                          // 4 consecutive columns can be stored as one vector
  int chain;                        // stages of a chain - 1 (a power of two less one)
};

template <typename TO, int FQ>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(F32Args a) {
  constexpr int BP = 64, BQ = 16 * FQ, GW = BP / 32, GX = (FQ + 1) / 2, G = GW + GX, STAGE = 32 * G * 128;
  constexpr int NS = FQ > 4 ? 3 : 4;                       // 72 KB at most: two workgroups on a CU
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) char lds[NS * STAGE];
  // blocks of one XCD (id % 8) take consecutive tiles, rows fastest: a column's weights are read from one L2
  const int tot = a.mt * a.nt * a.batch, q8 = tot >> 3, r8 = tot & 7, xcd = blockIdx.x & 7;
  int t = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (int)(blockIdx.x >> 3);
  const int ti = t % a.mt;
  t /= a.mt;
  const int tj = t % a.nt, tb = t / a.nt;
  const float *A = a.A + (size_t)tb * a.sA, *W = a.W + (size_t)tb * a.sW;
  int row0 = ti * BQ, rows = min(BQ, a.M - row0);
  if (a.tiles != nullptr) {
    constexpr int PER = 64 / BQ > 0 ? 64 / BQ : 1;
    const int y = ti / PER, sub = (ti - y * PER) * BQ, g = a.tiles[3 * y];
    if (g < 0) return;
    row0 = a.tiles[3 * y + 1] + sub;
    rows = min(BQ, a.tiles[3 * y + 2] - sub);
    if (rows <= 0) return;
    W += (size_t)g * a.sW;
  }
  const int col0 = tj * BP;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, g = lane >> 4;
  // loader: instruction j moves the stage's rows 32 j .. 32 j + 31 (weights first), 16 bytes a thread; rows past the end
  // repeat the last one
  const float* src[G];
  const int lr = tid >> 3, lc = ((tid & 7) ^ (lr & 7)) * 4;
#pragma unroll
  for (int j = 0; j < G; ++j) {
    if (j < GW) {
      src[j] = W + (size_t)min(col0 + 32 * j + lr, a.N - 1) * a.ldw + lc;
    } else {
      const int r = row0 + min(32 * (j - GW) + lr, rows - 1);
      src[j] = A + (size_t)(a.a_rows != nullptr ? a.a_rows[r] : r) * a.lda + lc;
    }
  }
  auto dma = [&](int u, int slot, int j) {
    __builtin_amdgcn_global_load_lds(src[j] + (size_t)u * 32,
                                     (__attribute__((address_space(3))) void*)(lds + slot * STAGE + wid * 1024 + j * 4096),
                                     16, 0, 0);
  };
  const uint32_t base = (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)lds);
  const uint32_t pw = base + (wid * 16 + li) * 128, px = base + (BP + li) * 128;
  const uint32_t ch[2] = {(uint32_t)(g ^ (li & 7)) << 4, (uint32_t)((4 + g) ^ (li & 7)) << 4};
  f32x4 w0, w1, x0[FQ], x1[FQ], acc[FQ], sum[FQ];
#pragma unroll
  for (int j = 0; j < FQ; ++j) sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Reads and products are volatile asm in program order (as in pgemm4.hip): the compiler does not drain the LDS counter
  // ahead of every product.  Nothing touches a fragment before the lgkmcnt(0) that ends the phase of its read.
  auto read = [&](uint32_t o, int r, f32x4& w, f32x4* x) {
    if (r == 0) asm volatile("ds_read_b128 %0, %1" : "=v"(w) : "v"(pw + o));
    else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(x[r - 1]) : "v"(px + o), "i"((r - 1) * 2048));
  };
  // products of (wc, xc) -- `fresh`: onto zero -- with the reads at o into (wn, xn) in their first half, and in the second
  // (u >= 0) the loads of stage u into slot us
  auto phase = [&](auto fresh, const f32x4& wc, const f32x4* xc, f32x4& wn, f32x4* xn, uint32_t o, int u, int us) {
    constexpr int MF = 4 * FQ;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        const int k = e * FQ + j;
        if (decltype(fresh)::value && e == 0)
          asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, 0" : "=&v"(acc[j]) : "v"(wc[e]), "v"(xc[j][e]));
        else
          asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+v"(acc[j]) : "v"(wc[e]), "v"(xc[j][e]));
#pragma unroll
        for (int r = 0; r <= FQ; ++r)
          if (k == r * (MF / 2) / (FQ + 1)) read(o, r, wn, xn);
#pragma unroll
        for (int d = 0; d < G; ++d)
          if (k == MF / 2 + d * (MF / 2) / G && u >= 0) dma(u, us, d);
      }
  };
  auto landed = [&]() {       // every wave's part of the next stage is in LDS, and every read of the current one has retired
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    f32_vmcnt<(NS - 2) * G>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto flush = [&]() {        // the products are opaque to the hazard recogniser: their results wait out the latency first
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
    for (int j = 0; j < FQ; ++j) {
      asm volatile("" : "+v"(acc[j]));
      sum[j] += acc[j];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int S = a.K / 32;
#pragma unroll
  for (int q = 0; q < NS - 1; ++q)
#pragma unroll
    for (int d = 0; d < G; ++d) dma(min(q, S - 1), q, d);
  landed();
#pragma unroll
  for (int r = 0; r <= FQ; ++r) read(ch[0], r, w0, x0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  int slot = 0;
  for (int s = 0; s < S; ++s) {
    // stage s + NS - 1 (past the end: the last one again) goes into the slot of s - 1, whose reads every wave has retired
    const int us = slot == 0 ? NS - 1 : slot - 1, u = min(s + NS - 1, S - 1);
    const uint32_t o1 = (uint32_t)(slot * STAGE) + ch[1];
    if ((s & a.chain) == 0) phase(std::true_type{}, w0, x0, w1, x1, o1, u, us);
    else phase(std::false_type{}, w0, x0, w1, x1, o1, u, us);
    slot = slot + 1 == NS ? 0 : slot + 1;
    landed();
    phase(std::false_type{}, w1, x1, w0, x0, (uint32_t)(slot * STAGE) + ch[0], -1, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if ((s & a.chain) == a.chain || s == S - 1) flush();
  }
  f32_vmcnt<0>();             // no load into LDS is left behind
  // sum[j][e] = C[row 16 j + li][column 16 wid + 4 g + e]
  TO* C = reinterpret_cast<TO*>(a.C) + (size_t)tb * a.sC;
  const int c = col0 + 16 * wid + 4 * g;
#pragma unroll
  for (int j = 0; j < FQ; ++j) {
    const int r = 16 * j + li;
    if (r >= rows || c >= a.N) continue;
    const size_t at = (size_t)(row0 + r) * a.ldc + c;
    if (a.vec) {
      stf4(C + at, sum[j]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < a.N) stf(C, at + e, sum[j][e]);
    }
  }
#endif
}

// The same product with k shared by the waves instead of the columns: a wave owns all 64 columns x 16 FQ rows of the tile for a
// quarter of k, stages its own weights and rows (16-deep, 64-byte rows, a ring of 4 slots) and meets the others once, at the
// end, in LDS -- no barrier and no other wave's loads to wait for while k lasts.  85 - 90 % of the matrix rate on a CU with one
// workgroup (all that the rings leave room for, but at FQ = 1, where two fit).  us, columns shared -> k shared:
// 333 x 2048 x 2048 35.0 -> 31.4, x 8192 129 -> 109, 200 x 2048 x 8192 97 -> 79, 200 x 4096 x 4096 81 -> 73,
// 100 x 4096 x 14336 170 -> 144, 64 x 16384 x 2048 50 -> 45; in three rounds and more it is behind (333 x 16384 x 2048 180 and 203).  Ahead of gemm_f32_kernel's eight shares too: 333 x 576 x 2048
// 18.0 -> 14.4, 64 x 2048 x 8192 68 -> 58.  Error against 64 bits, 2-norm: 2.1e-7 - 2.3e-7.
template <typename TO, int FQ>
__global__ __launch_bounds__(256, 1) void gemm_f32_kwave_kernel(F32Args a) {
  constexpr int BP = 64, BQ = 16 * FQ, G = 4 + FQ, STAGE = G * 1024, NS = 4, RING = NS * STAGE;
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) char lds[4 * RING];
  static_assert(4 * RING >= 4 * BP * BQ * 4, "the waves' sums fit the rings");
  const int tot = a.mt * a.nt * a.batch, q8 = tot >> 3, r8 = tot & 7, xcd = blockIdx.x & 7;
  int t = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (int)(blockIdx.x >> 3);
  const int ti = t % a.mt;
  t /= a.mt;
  const int tj = t % a.nt, tb = t / a.nt;
  const float *A = a.A + (size_t)tb * a.sA, *W = a.W + (size_t)tb * a.sW;
  int row0 = ti * BQ, rows = min(BQ, a.M - row0);
  if (a.tiles != nullptr) {
    constexpr int PER = 64 / BQ > 0 ? 64 / BQ : 1;
    const int y = ti / PER, sub = (ti - y * PER) * BQ, g = a.tiles[3 * y];
    if (g < 0) return;
    row0 = a.tiles[3 * y + 1] + sub;
    rows = min(BQ, a.tiles[3 * y + 2] - sub);
    if (rows <= 0) return;
    W += (size_t)g * a.sW;
  }
  const int col0 = tj * BP;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, g = lane >> 4;
  const int S = a.K / 16, first = wid * S / 4, last = (wid + 1) * S / 4 - 1;     // this wave's 16-deep stages (K >= 64)
  // loader: instruction j moves 16 rows of the stage (weights first), 16 bytes a lane; rows past the end repeat the last one
  const float* src[G];
  const int lr = lane >> 2, lc = ((lane & 3) ^ (lr >> 2)) * 4;
#pragma unroll
  for (int j = 0; j < G; ++j) {
    if (j < 4) {
      src[j] = W + (size_t)min(col0 + 16 * j + lr, a.N - 1) * a.ldw + lc;
    } else {
      const int r = row0 + min(16 * (j - 4) + lr, rows - 1);
      src[j] = A + (size_t)(a.a_rows != nullptr ? a.a_rows[r] : r) * a.lda + lc;
    }
  }
  char* mine = lds + wid * RING;
  auto dma = [&](int u, int slot, int j) {
    __builtin_amdgcn_global_load_lds(src[j] + (size_t)u * 16,
                                     (__attribute__((address_space(3))) void*)(mine + slot * STAGE + j * 1024), 16, 0, 0);
  };
  const uint32_t base = (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)mine);
  const uint32_t pl = base + li * 64 + ((g ^ (li >> 2)) << 4);
  f32x4 f0[G], f1[G], acc[4][FQ], sum[4][FQ];      // fragments: 4 of weights, FQ of rows
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < FQ; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto read = [&](uint32_t o, int r, f32x4* f) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f[r]) : "v"(pl + o), "i"(r * 1024));
  };
  // Products of f with (more) the reads of the next stage at o into n in their first half and the loads of stage u into slot us,
  // whose fragments are those of f, in the second.  A read's output is always used by the next phase, and nothing touches it
  // before the wait at the end; the products are opaque to the hazard recogniser, so the phase also waits out their latency
  // (the matrix unit is busy with the last one that long anyway).
  auto phase = [&](auto more, const f32x4* f, f32x4* n, uint32_t o, int u, int us) {
    constexpr int MF = 16 * FQ;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < FQ; ++j) {
          const int k = (e * 4 + i) * FQ + j;
          asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(f[i][e]), "v"(f[4 + j][e]));
          if constexpr (decltype(more)::value) {
#pragma unroll
            for (int r = 0; r < G; ++r)
              if (k == r * (MF / 2) / G) read(o, r, n);
#pragma unroll
            for (int d = 0; d < G; ++d)
              if (k == MF / 2 + d * (MF / 2) / G) dma(u, us, d);
          }
        }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    if constexpr (decltype(more)::value) f32_vmcnt<(NS - 2) * G>();        // the stage after the next has landed
    __builtin_amdgcn_sched_barrier(0);
  };
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+v"(acc[i][j]));
      }
    asm volatile("s_nop 7" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto flush = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        asm volatile("" : "+v"(acc[i][j]));
        sum[i][j] += acc[i][j];
      }
    clear();
  };
#pragma unroll
  for (int q = 0; q < NS; ++q)
#pragma unroll
    for (int d = 0; d < G; ++d) dma(min(first + q, last), q, d);
  clear();
  f32_vmcnt<(NS - 1) * G>();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < G; ++r) read(0, r, f0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  f32_vmcnt<(NS - 2) * G>();
  __builtin_amdgcn_sched_barrier(0);
  const int n = last - first + 1, chain = 2 * a.chain + 1;        // a chain's stages - 1
  int slot = 0, s = 0;
  auto step = [&](auto more, const f32x4* f, f32x4* nx) {
    const int next = slot + 1 == NS ? 0 : slot + 1;
    phase(more, f, nx, (uint32_t)(next * STAGE), min(first + s + NS, last), slot);
    slot = next;
    if ((s & chain) == chain || !decltype(more)::value) flush();
    ++s;
  };
  constexpr std::true_type yes{};
  while (s + 2 < n) {
    step(yes, f0, f1);
    step(yes, f1, f0);
  }
  if (s + 2 == n) {
    step(yes, f0, f1);
    step(std::false_type{}, f1, f0);
  } else {
    step(std::false_type{}, f0, f1);
  }
  f32_vmcnt<0>();             // no load into LDS is left behind
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < FQ; ++j) *reinterpret_cast<f32x4*>(red + (((wid * 4 + i) * FQ + j) * 64 + lane) * 4) = sum[i][j];
  __syncthreads();
  // C[row 16 j + li][column 16 wid + 4 g + e]
  TO* C = reinterpret_cast<TO*>(a.C) + (size_t)tb * a.sC;
  const int c = col0 + 16 * wid + 4 * g;
#pragma unroll
  for (int j = 0; j < FQ; ++j) {
    const int r = 16 * j + li;
    f32x4 y = *reinterpret_cast<const f32x4*>(red + ((wid * FQ + j) * 64 + lane) * 4);
#pragma unroll
    for (int w = 1; w < 4; ++w) y += *reinterpret_cast<const f32x4*>(red + (((w * 4 + wid) * FQ + j) * 64 + lane) * 4);
    if (r >= rows || c >= a.N) continue;
    const size_t at = (size_t)(row0 + r) * a.ldc + c;
    if (a.vec) {
      stf4(C + at, y);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < a.N) stf(C, at + e, y[e]);
    }
  }
#endif
}

}  // namespace k8sllm

using namespace k8sllm;

// The tile for a product (0: gemm_f32_kernel's are expected to be as good); 16 more: k shared by the waves.  Whether, and which of the
// two, in us per 32 k, one constant part and one per round of tiles over the CUs, fitted to M 24 - 512, N 128 - 16384, K 512 - 8192 (where
// the two models are within 5 % of each other, so are the kernels); a round of one workgroup per CU with k shared also pays its start and
// its sum (4.5 us, of which nothing overlaps), so that is the choice for one or two rounds.  Where columns are faster there all the same
// (28672 x 4096, 24 - 64 rows, 116 / 95 and 156 / 149 us; 384 x 4096 x 4096 117 / 112) the shares keep the smaller error, 2-norm against 64
// bits: K = 4096 2.15e-7 / 2.29e-7, 14336 2.3e-7 / 2.8e-7.
// How many rows a tile of columns has goes by a fit of 8 shapes of 2048 x 2048 .. 28672 x 4096, rms error 4 %: a part per round, one for
// an odd round of up to three (its tiles are alone on their CUs) and one a product; from eight rounds on one that is partly filled costs that
// part.  By the first fit / this one: 457 x 6720 x 4096 276 / 255, 441 x 3072 x 1536 50 / 47, 384 x 3648 x 2048 58.0 / 56.8, 393 x 14336 x
// 4096 429 / 417; without the two exceptions 401 x 6144 x 4096 195 / 182, 352 x 7168 x 4096 195 / 183.  K < 512: shares of K / 8 leave the
// smaller error.
static int f32_rule(int M, int N, int K, int batch, int ntiles, double* cost) {
  *cost = 0.0;
  if (K < 512 || K % 32 || M <= 0 || N <= 0) return 0;
  // Listed tiles: most of the list is short of 64 rows or empty, and where its blocks meet on a CU is left to chance, so the parts
  // below do not hold.  From 32 rows a group on (the list has one tile a group more than the rows fill) 32-row tiles, where the
  // 64-row ones would be 280 and more, and from 1000 of 64 rows and more a group on those.  us, gemm_f32_kernel / 32 / 64 rows,
  // weights from memory, groups x columns x k, rows a group: 8 x 4096 x 2048, 24 63 / 87 / 81, 40 100 / 86 / 80, 96 162 / 149 /
  // 142; 8 x 2048 x 2048, 24 54 / 60 / 72, 40 61 / 58 / 71, 130 115 / 103 / 109; 16 x 1024 x 2048, 40 61 / 46 / 72, 500 352 / 303 / 307;
  // 4 x 2048 x 2048 (144 tiles), 40 32 / 42 / 43.
  if (ntiles > 0) {
    const long groups = ntiles - (M + 63) / 64 > 1 ? ntiles - (M + 63) / 64 : 1;
    const double t = (M / 64.0 + groups / 2.0) * ((N + 63) / 64);
    return M < 32 * groups || t < 280.0 ? 0 : M >= 64 * groups && t >= 1000.0 ? 4 : 2;
  }
  const auto rounds = [&](long rows, long cols) { return (double)((rows * cols * batch + 255) / 256); };
  const long gm = (M + 31) / 32;
  const double r1 = rounds(gm, (N + 31) / 32), r2 = rounds(gm, (N + 63) / 64);
  // Few rows in one round of gemm_f32_kernel's tiles wait for weights that none but their own workgroup reads, which the fitted
  // parts leave out; the tiles of 64 columns keep fewer CUs loading.  us, k shared by the waves / gemm_f32_kernel, weights from
  // memory: 1 row, 2048 x 2048 19.3 / 19.2, 4096 x 14336 135 / 120; 16 rows 22.8 / 19.6, 155 / 120; narrow ones, 128 x 2048, 1 row
  // 17.7 / 18.5, 4 rows 19.0 / 18.6, 16 rows 21.8 / 19.0 (from the cache 13.5 / 16.7).  From 17 rows on two row tiles share them:
  // 17 rows 18.5 / 19.6, 2048 x 8192 61.5 / 68.7, 4096 x 14336 124 / 120; 24 rows 20.0 / 19.7, 67.1 / 68.7, 129 / 121; 32 rows
  // 20.8 / 19.8, 70.1 / 68.7.
  const long cols = (long)N * batch;
  // us, from the fitted parts: a constant, so much of the parts, and a share of what the weights take
  const auto us = [&](double c, double parts, double weights) { *cost = c + parts * K / 32.0 + weights * 4e-6 * cols * (double)K; };
  if (r1 == 1.0 && M <= 32 && (M <= 4 ? cols > 256 : M <= 16 || M > 24 || cols > 2048)) {
    us(3.0, 0.787 * 0.26, 0.101);
    return 0;
  }
  double best = 2.0 * r2 < 1.1 * r1 ? 0.365 * r2 + 0.03 : 0.16 * r1 + 0.1;
  int pick = 0;
  for (int fq = 8; fq >= 1; --fq) {
    const double r = rounds((M + 16 * fq - 1) / (16 * fq), (N + 63) / 64);
    const double t = r * (0.125 * fq + 0.04) + 0.1;
    if (t < best) {
      best = t;
      pick = fq;
    }
    const double tk = r * (0.12 * fq + 0.03 + 4.5 * 32 / K);
    if (fq <= 4 && tk < 0.96 * best) {
      best = tk;
      pick = 16 + fq;
    }
  }
  if (pick == 0) us(2.1, 1.052 * best, 0.156);
  else if (pick > 16) us(0.0, 1.044 * best, 0.078);
  if (pick == 0 || pick > 16) return pick;
  best = 1e30;
  for (int fq = 8; fq >= 1; --fq) {
    const double tiles = (double)((M + 16 * fq - 1) / (16 * fq)) * ((N + 63) / 64) * batch / 256.0, r = ceil(tiles);
    const double t = (r >= 8.0 ? tiles : r) * (0.1157 * fq + 0.056) + (r == 1.0 || r == 3.0 ? 0.002 * fq + 0.0666 : 0.0);
    if (t < best) {
      best = t;
      pick = fq;
    }
  }
  us(4.1, 1.108 * best, 0.039);
  return pick;
}

extern "C" int k8s_gemm_f32_rule(int M, int N, int K, int batch, int ntiles) {
  double cost;
  return f32_rule(M, N, K, batch, ntiles, &cost);
}

// What a product of K >= 512 takes on the fp32 pipes by that choice, us (fitted to M 1 - 512, N 128 - 32768, K 512 - 14336; rms error 3 - 8 %)
extern "C" double k8s_gemm_f32_cost(int M, int N, int K, int batch) {
  double cost;
  f32_rule(M, N, K, batch, 0, &cost);
  return cost;
}

// fq: rows of a tile / 16 (1 - 8; listed tiles of at most 64 rows: 1, 2, 4), or 16 + that (1 - 4): k shared by the waves.
extern "C" int k8s_gemm_f32_tiles(void* C, const float* A, const float* W, int M, int N, int K, long lda, long ldw, long ldc,
                                  int batch, long sA, long sW, long sC, const int* a_rows, const int* tiles, int ntiles,
                                  int out_f32, int fq, hipStream_t s) {
  const bool kwave = fq > 16;
  if (kwave) fq -= 16;
  if (M <= 0 || N <= 0 || K < (kwave ? 64 : 32) || K % 32 || batch <= 0 || fq < 1 || fq > (kwave ? 4 : 8) || (lda | ldw | sA | sW) % 4 ||
      (((uintptr_t)A | (uintptr_t)W) & 15))
    return -1;
  if (tiles != nullptr && (64 % (16 * fq) || ntiles <= 0)) return -1;
  F32Args a = {C, A, W, M, N, K, 0, 0, 0, lda, ldw, ldc, sA, sW, sC, a_rows, tiles, 0};
  a.mt = tiles != nullptr ? ntiles * (4 / fq) : (M + 16 * fq - 1) / (16 * fq);
  a.nt = (N + 63) / 64;
  a.batch = tiles != nullptr ? 1 : batch;
  const long long blocks = (long long)a.mt * a.nt * a.batch;
  if (blocks > (1LL << 30)) return -2;
  a.vec = N % 4 == 0 && ldc % 4 == 0 && sC % 4 == 0 && ((uintptr_t)C & 15) == 0;
  a.chain = K >= 2048 ? 3 : K >= 1024 ? 1 : 0;
  auto go = [&](auto n) {
    constexpr int FQ = decltype(n)::value;
    if constexpr (FQ <= 4) {
      if (kwave) {
        if (out_f32) gemm_f32_kwave_kernel<float, FQ><<<dim3((unsigned)blocks), 256, 0, s>>>(a);
        else gemm_f32_kwave_kernel<bf16_t, FQ><<<dim3((unsigned)blocks), 256, 0, s>>>(a);
        return;
      }
    }
    if (out_f32) gemm_f32_tile_kernel<float, FQ><<<dim3((unsigned)blocks), 256, 0, s>>>(a);
    else gemm_f32_tile_kernel<bf16_t, FQ><<<dim3((unsigned)blocks), 256, 0, s>>>(a);
  };
  switch (fq) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
  }
  return (int)hipGetLastError();
}
