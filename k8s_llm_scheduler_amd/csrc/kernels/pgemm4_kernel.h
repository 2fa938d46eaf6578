// The kernel of pgemm4.hip, its tile configurations and their launches; pgemm4.hip, pgemm4_tiles.hip and pgemm4_wide.hip instantiate a
// part of the tiles each.
//
// K3 / K8 / K9(+K10) / K11 / K12 at prefill row counts, bf16: the 4-wave big-tile MFMA GEMM.
//
//     out[M, N_out] = epi( x[M, K] . W[N, K]^T )      epi: bf16 (+ residual) | fp32 | SwiGLU, optional RMS prologue;
//                                                     an activation (elementwise, or gated with W = [gate; up])
//
// Why 4 waves (and not pgemm.hip's 8-wave ping-pong): PMC on the 2048 x 8192 x 8192 projection showed the
// 8-wave 128 x 64-per-wave schedule parked 31 % of its wave cycles at barriers (SQ_WAIT_ANY) and issued 1.5x
// the LDS instructions of the library's 256 x 256 kernel, which runs 4 waves of 128 x 128
// (profiles/pmc_pgemm_vs_hipblaslt_M2048_oproj_tp1.txt).  Here every wave owns a 128 x 128 output (64
// fragments of v_mfma_f32_16x16x32_bf16, 256 accumulator registers: the AGPR half of the unified file at one
// wave per SIMD), so per 32 k a wave issues 16 fragment reads for 64 MFMAs.
//
//  * 64-deep LDS stages of 128-byte rows (every LDS-DMA instruction moves 8 whole rows), DW stages of weights and DX of x in
//    flight across the raw s_barriers, of which there is one per 2 x FP x FQ MFMAs: two and one (three slots, two) from 128 x 64
//    on -- all of the CU's 160 KB at 256 x 256, two workgroups on a CU at 128 x 128, where more of them measured 0 - 5 % -- and four of
//    both at 64 x 64, whose stage is 0.1 us of matrix work against a load's 0.5 - 2 (200 x 2048 x 2048 12.6 -> 9.5 us, 333 x 2128 x 2048
//    0.66 of its time; two workgroups on a CU still).  The least that a stage can take: 32 KB of the two operands in 0.26 us out of
//    L2 (53 bytes a cycle and CU), what misses L2 at 6 - 7 TB/s whatever holds it.
//  * one row tile (the weights are read once): XCD i starts its walk over k at stage i n / 8 and wraps.  In step with each other
//    all of them ask for the same bytes of every row, whose strides of 16 KB meet on a part of the memory's channels, and for the
//    same lines of x (loads alone, 32768 rows of 16 KB: 4.1 -> 6 TB/s).  241 x 57344 x 8192 251 -> 230 us, 8192 x 28672 136 -> 131,
//    8192 x 8192 50 -> 47.  With more row tiles the walk in step is the better one (2048 x 16384 x 2048 106 -> 111): so not there; the
//    grouped form by its rows (P4Args::spread); but deep ones, whose rows' strides put whole columns of tiles on the same channels, from
//    16384 columns on up to 8 row tiles, which then follow each other (group_m): 7 weights of 4096 - 16384 x 16384 - 28672, 333 - 2048 rows,
//    12 % less time with 2 row tiles, 5 - 8 % with 3 - 7, 3 % with 8 (at most 5 % more, on 5120 x 20480 with 8); 8192 x 28672, 333 rows 164 ->
//    152 us, 1536 525 -> 490; 12288 x 24576, 333 237 -> 192.  In groups of 4, 6 and 8 row tiles were 1 % slower than in step, in groups of 2 1 - 4 %
//    whatever their number.  3413 rows of 8192 x 28672 1265 -> 1279; of 14336 columns and fewer 1 % slower on average.
//  * rows of 4 KB and less (K up to 2048) on tiles of at most 128 x 128 and on those of 32 tokens: every column of tiles starts its walk
//    an eighth of it after the one before (P4Args::fine): at one k the rows' bytes lie in a few of the memory's channels, and short
//    tiles have no time to drift apart.  us: 2048 x 2048 x 2048 21.1 -> 19.0, 1024 x 3072 x 2048 19.1 -> 16.3, 512 x 3648 x 2048 16.4 ->
//    13.2, gated 130 x 2 x 8192 x 2048 26.6 -> 25.3; over 65 products of 128 - 3413 rows 3 - 5 % less on average, none more than 1.8 % slower.  Of
//    larger tiles, which read x from L2 in step, 2 - 12 % slower; of K = 4096 at 128 x 128 0.89 - 1.20 of the time.
//  * tiles of 224 rows (a fragment then holds 8 gate and 8 up rows, a pair in a lane) and of 192 tokens, where they fill the last
//    round: 241 x 57344 x 8192 on 256 CUs 230 -> 207 us, 3413 x 10240 x 8192 484 -> 412.
//  * register double buffer: the fragments of the next 32 k are read (ds_read_b128) under the MFMAs of the current ones, in
//    the first half of them: spread over all of them, the wait at the end stood 100 - 150 of 1024 matrix cycles a step.
//  * DMA image lane-linear, XOR swizzle on the per-lane global source: the 16-row fragment reads are conflict-free.
//  * bf16 output through LDS, in 64 - 256-byte runs of a row a store instead of 32-byte pieces of 16 rows.
//  * swapped orientation C^T = W . x^T: every lane ends with 4 consecutive features of one token (gate/up
//    rows of one feature sit in the same lane for the SwiGLU epilogue).
//  * XCD-aware bijective block remap, group_m m-tiles per n-column group, k-slices of a tile adjacent.
//  * split-K: every slice stores fp32 partial sums into its own slab [M][W rows] (plus the RMS row sums) and
//    pgemm_reduce_kernel sums the slabs in slice order (deterministic) and applies the epilogue -- a
//    parallel reduction over the whole chip instead of one last-arriving workgroup reading every slab.
//
// us, weights from memory (rows x N x K), with 32-deep stages, reads and stores spread as they fell -> as above, and hipBLASLt:
// 256 x 256 tiles 2048 x 8192 x 2048 64 -> 56 (52), x 8192 208 -> 188 (188), 3413 x 8192 x 8192 364 -> 342 (333); 128 x 256
// 2048 x 8192 x 2048 82 -> 64; 128 x 128 2048 x 2048 x 2048 25 -> 22 (22), x 8192 94 -> 73 (78).  Bound by the matrix rate at
// the clock that the power allows (1.7 - 2.0 GHz in long launches; operands all zero take 25 % less time): 89 % of a stage's
// cycles are the matrix cores', and at K = 2048 a fifth of the launch is its start, first loads and stores.  The 256 x 256 tiles
// take all 512 registers, and by the compiler's report spill 16 - 38 of them between the k loop and the rows in LDS (bf16 20,
// SwiGLU 31, fp32 output 0, with the RMS prologue 28, 24 and 12, with row scales 20 and 32; the gated kinds 26 - 38, relu^2 16), none
// of it inside the loop.
#pragma once

#include <type_traits>

#include "act.h"
#include "common.h"

namespace k8sllm {

namespace {
enum { P4_BF16 = 0, P4_F32 = 1, P4_SWIGLU = 2, P4_GLU = 3, P4_ACT = 4 };   // GLU, ACT: bf16 out, activation KIND
enum { P4_PLAIN = 0, P4_RMS = 1, P4_SCALED = 2 };   // rows as they are; 1 / rms from a prologue in the k loop; from P4Args::scale
typedef __attribute__((ext_vector_type(2))) uint32_t p4_u32x2;
typedef __attribute__((ext_vector_type(2))) float p4_f32x2;

template <int N>
__device__ __forceinline__ void p4_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void p4_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// LDS-DMA of 16 bytes a lane, from a uniform base and the lane's 32-bit offset to LDS byte `lds` + 16 lane.  In asm: from the
// builtin the compiler hoists base + offset, or the widened offset, into 64-bit lane addresses and adds the step to each of
// them, an instruction and two registers per load.  m0 is the compiler's own, which it need not keep for itself across an asm that
// names it (the warning that is off here): nothing else in this file may want it -- no LDS-DMA builtin, no register indexed at run
// time.  (In this file's assembly every m0 is the move of one of these.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void p4_dma(const uint8_t* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ float p4_silu(float g) { return g / (1.f + __expf(-g)); }
// The kind of an activation (act.h) is a template argument: 128 unrolled elements per lane with every kind's branches took 775
// us where the product takes 56.
}  // namespace

struct P4Args {
  void* out;
  const bf16_t* res;     // optional residual (bf16 [M][N_out], may alias out)
  float* slab;           // split-K: [splits][M][W rows] fp32 partial sums, then [splits][M] row sums of squares
  const uint8_t* x;      // [M][K] bf16
  const uint8_t* W;      // [rows][K] bf16
  uint32_t kbytes;       // bytes per row of x and W
  uint32_t xbytes;       // grouped form: bytes per row of x
  int M, N_out, half_rows, wrows, K;
  int m_tiles, n_tiles, ks, splits, group_m, nwg;
  float eps;
  const float* scale;    // P4_SCALED: 1 / rms of every token's row
  int spread;            // the XCDs start their walk over k an eighth of it apart
  int fine;              // ... and the tile columns fine / 32 of it, on top of that
  int wide;              // the output's rows can be stored in 16-byte pieces
  float limit, alpha;    // P4_GLU: of the gated kind
  float last_limit;      // grouped form: the limit of the last group
  const bf16_t* bias;    // P4_GLU, optional: [gate; up] biases
  // grouped form: group g's rows are [seg[g], seg[g + 1]) of a compact row space (row r of x: a_rows[r], or r) and its
  // weights W + g wstride bytes; m_tiles bounds the groups' row tiles.  8 experts, 3068 rows, K = 2048, in a step, as it was
  // brought here: gate / up with its activation (N = 2 x 2048) 69 us, down (N = 2048) 34 us; on the 64-row tiles of stream32.hip 140 and
  // 10 us, and 78 us.
  // spread with 8 groups and more, an XCD's tiles then another group's, of up to 192 rows: gate / up of 8 experts, 4 - 192 rows
  // each 29.4 -> 27.8 us (64 x 64), 16 of 2 x 2048 x 4096 139 -> 108 (256 x 128); 4 groups 30.0 -> 34.0, 320 rows 70 -> 71.
  // seg == nullptr: groups of gsize rows (products of several inputs with a weight each in one launch)
  const int* seg;
  int gsize;
  const int* a_rows;
  long long wstride;
  int groups;
};

template <int FP, int FQ, int DW, int DX, int EPI, int NORM, bool GRP = false, int KIND = -1>
__global__ void __launch_bounds__(256, 1) pgemm4_kernel(P4Args a) {
  constexpr bool RMS = NORM == P4_RMS;
  static_assert(DW == DX || DW == DX + 1, "a stage's last load is followed by whole stages of later ones");
  constexpr int BP = 32 * FP, BQ = 32 * FQ;          // weight rows, tokens per tile (2 x 2 waves)
  constexpr bool PAIR = EPI == P4_SWIGLU || EPI == P4_GLU;   // gate and up rows of one feature in one wave
  constexpr bool MIX = PAIR && FP % 2 != 0;          // ... and in one fragment: a lane's four rows are gate, gate, up, up
  static_assert(!GRP || NORM == P4_PLAIN, "the grouped form has no prologue");
  constexpr int SUBW = BP * 128, SUBX = BQ * 128;    // a 64-deep stage of either operand
  constexpr int GW = BP / 32, GX = BQ / 32;          // 16-byte DMA instructions per thread and stage
  constexpr int X0 = (DW + 1) * SUBW, RING = X0 + (DX + 1) * SUBX;
  constexpr int RSS = RING - BQ * 8;                 // in the last stage's memory, once it has been read
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) char lds[RING];
  float* rss = reinterpret_cast<float*>(lds + RSS);   // [2][BQ] row sums of squares (wave rows)

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid >> 1, wc = wid & 1;
  const int li = lane & 15, g = lane >> 4;

  // ---- block -> (tile, k-slice)
  int nwg = a.nwg, m_tiles = a.m_tiles;
  auto first = [&](int e) { return a.seg != nullptr ? a.seg[e] : e * a.gsize; };   // group e's first row
  if constexpr (GRP) {     // the launch covers an upper bound: spread the tiles there are over the XCDs
    m_tiles = 0;
    for (int e = 0; e < a.groups; ++e) m_tiles += (first(e + 1) - first(e) + BQ - 1) / BQ;
    nwg = m_tiles * a.n_tiles;
    if ((int)blockIdx.x >= nwg) return;
  }
  const int bid = blockIdx.x, q8 = nwg >> 3, r8 = nwg & 7, xcd = bid & 7, loc = bid >> 3;
  const int lid = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + loc;
  const int tile = lid / a.splits, slice = lid - tile * a.splits;
  int mt, nt;
  {
    const int per = a.group_m * a.n_tiles, gi = tile / per, mg = gi * a.group_m;
    const int gm = min(m_tiles - mg, a.group_m), in = tile - gi * per;
    mt = mg + in % gm;
    nt = in / gm;
  }
  // tokens of the tile: rows [m0, m_end) of the compact row space
  const uint8_t* Wb = a.W;
  int m0 = mt * BQ, m_end = a.M;
  float limit = a.limit;
  if constexpr (GRP) {
    int gi = 0, left = mt;                           // mt < m_tiles: a group is found
    for (;; ++gi) {
      const int nt_g = (first(gi + 1) - first(gi) + BQ - 1) / BQ;
      if (left < nt_g) break;
      left -= nt_g;
    }
    m0 = first(gi) + left * BQ;
    m_end = first(gi + 1);
    Wb += (long long)gi * a.wstride;
    if (gi == a.groups - 1) limit = a.last_limit;
  }
  auto xrow = [&](int r) -> uint32_t {               // row r of the tile, past the end its last one
    const int m = min(m0 + r, m_end - 1);
    if constexpr (GRP) return (uint32_t)(a.a_rows != nullptr ? a.a_rows[m] : m);
    return (uint32_t)m;
  };
  const int ks0 = 2 * (int)((long long)slice * (a.ks / 2) / a.splits);
  const int n2 = (int)((long long)(slice + 1) * (a.ks / 2) / a.splits) - ks0 / 2;   // 64-deep stages, >= 1

  // ---- per-thread DMA sources: chunk p = j * 256 + tid of the stage image, 8 chunks of 16 bytes a row
  const uint32_t col0 = (uint32_t)(ks0 * 64);
  uint32_t wo[GW], xo[GX];
#pragma unroll
  for (int j = 0; j < GW; ++j) {
    const int p = j * 256 + tid, r = p >> 3, c = (p & 7) ^ ((r >> 1) & 7);
    const int w = r / (BP / 2), q = r % (BP / 2);
    int row;
    if constexpr (MIX) {
      const int f = min(nt * (BP / 2) + w * (BP / 4) + (q >> 4) * 8 + ((q >> 1) & 6) + (q & 1), a.N_out - 1);
      row = q & 2 ? a.half_rows + f : f;
    } else if constexpr (PAIR) {   // wave rows: BP/4 gate rows then the matching BP/4 up rows
      const int f = min(nt * (BP / 2) + w * (BP / 4) + (q % (BP / 4)), a.N_out - 1);
      row = q < BP / 4 ? f : a.half_rows + f;
    } else {
      row = min(nt * BP + r, a.N_out - 1);
    }
    wo[j] = (uint32_t)row * a.kbytes + (uint32_t)(c * 16) + col0;
  }
#pragma unroll
  for (int j = 0; j < GX; ++j) {
    const int p = j * 256 + tid, r = p >> 3, c = (p & 7) ^ ((r >> 1) & 7);
    xo[j] = xrow(r) * (GRP ? a.xbytes : a.kbytes) + (uint32_t)(c * 16) + col0;
  }
  // this wave's 1 KB of the first 4 KB of LDS
  const uint32_t lds0 = (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)lds) + wid * 1024;
  // the walk over k starts at stage `rot` and wraps: stage u reads bytes k0(u) .. k0(u) + 127 of the slice's rows
  const int rot = a.spread ? (int)((((uint32_t)(4 * xcd + a.fine * nt) & 31u) * (uint32_t)n2) >> 5) : 0;
  const uint32_t kend = (uint32_t)n2 * 128u;
  auto next_k = [&](uint32_t k) -> uint32_t { return k + 128u == kend ? 0u : k + 128u; };
  // instruction d of a stage's weights (k offset, byte offset of its slot), of its x
  auto dma_w = [&](uint32_t k, int slot, int d) { p4_dma(Wb + k, wo[d], lds0 + slot + d * 4096); };
  auto dma_x = [&](uint32_t k, int slot, int d) { p4_dma(a.x + k, xo[d], lds0 + X0 + slot + d * 4096); };

  bf16x8 A0[FP], B0[FQ], A1[FP], B1[FQ];
  f32x4 acc[FP][FQ];
  float ss[FQ];
#pragma unroll
  for (int f = 0; f < FQ; ++f) ss[f] = 0.f;

  auto squares = [&](const bf16x8* B, bool sq) {
    if constexpr (RMS) {
      if (sq) {   // the two wave rows hold the same x fragments: each squares every other k-step
#pragma unroll
        for (int f = 0; f < FQ; ++f)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bf16x2 v2 = {B[f][2 * e], B[f][2 * e + 1]};
            ss[f] = __builtin_amdgcn_fdot2_f32_bf16(v2, v2, ss[f], false);
          }
      }
    }
  };
  // Called with the first k-steps' loads in flight (the zero comes out of an asm behind them, 256 register writes would
  // otherwise go first).  The inline-asm MFMAs are opaque to the hazard recognizer: every zeroed accumulator passes through
  // an asm tied to it after its write, all before the first MFMA (volatile asm keeps its order).
  auto clear = [&]() {
    float z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
      for (int j = 0; j < FQ; ++j) acc[i][j] = f32x4{z, z, z, z};
    asm volatile("s_nop 1" ::: "memory");
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
      for (int j = 0; j < FQ; ++j) asm volatile("s_nop 0" : "+a"(acc[i][j]));
  };
  // ---- 64-deep stages: weights of stage u in slot u % (DW + 1), x in slot u % (DX + 1); row r at r * 128 bytes, 16-byte chunk c of row
  // r at slot c ^ ((r >> 1) & 7) (the swizzle is applied on the per-lane global source, the DMA image is lane-linear).
  // Sub-step h (k 32 h .. 32 h + 31) of a fragment row li = chunks 4 h + g.  Register sets: R0 = (A0, B0) holds
  // sub-step 0, R1 = (A1, B1) sub-step 1.  Per stage s after the barrier: phase A = the MFMAs of (s - 1, 1) on R1
  // with the reads of (s, 0) into R0, the LDS-DMA of x of stage s + DX and then of the weights of stage s + DW (into the
  // slots of s - 1, whose reads every wave retired before the barrier) spread between them; phase P = the MFMAs of (s, 0)
  // on R0 with the reads of (s, 1) into R1.  The wait of a stage leaves what was issued behind it outstanding.
  // The fragment reads go out in the first half of a phase: at its end, where they had been spread to, the wait for them
  // stood 100 - 150 of 1024 matrix cycles per phase (8192 columns, 2048 rows, all operands zero: K = 8192 160 -> 140 us).
  const int lo0 = li * 128 + ((g ^ (li >> 1)) << 4), lo1 = li * 128 + (((4 + g) ^ (li >> 1)) << 4);
  const int pb2 = wr * (BP / 2) * 128, qb2 = X0 + wc * (BQ / 2) * 128;
  auto laddr = [&](int off) {
    return (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)(lds + off));
  };
  auto rd2 = [&](bf16x8* A, bf16x8* B) {   // (0, 0), not interleaved
    const uint32_t la = laddr(pb2 + lo0), lb = laddr(qb2 + lo0);
#pragma unroll
    for (int f = 0; f < FP; ++f) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(A[f]) : "v"(la), "i"(f * 2048));
#pragma unroll
    for (int f = 0; f < FQ; ++f) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(B[f]) : "v"(lb), "i"(f * 2048));
  };
  // the MFMAs on (Ac, Bc) with (rd) the reads of sub-step h of a stage (slots at lw, lx) into (An, Bn), (dx) the loads of x of
  // the stage at kx into the slot at px and (dw) of the weights of the one at kw into pw spread between them
  auto phase = [&](const bf16x8* Ac, const bf16x8* Bc, int lw, int lx, int h, bf16x8* An, bf16x8* Bn, uint32_t kw, int pw,
                   uint32_t kx, int px, auto rdc, auto dxc, auto dwc) {
    constexpr int MF = FP * FQ, DR = FP + FQ;
    constexpr bool rd = decltype(rdc)::value, dx = decltype(dxc)::value, dw = decltype(dwc)::value;
    const uint32_t la = laddr(lw + pb2 + (h ? lo1 : lo0)), lb = laddr(lx + qb2 + (h ? lo1 : lo0));
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        const int k = i * FQ + j;
#pragma unroll
        for (int d = 0; d < (GW + GX); ++d)
          if (k == d * MF / (GW + GX)) {
            if (d < GX && dx) dma_x(kx, px, d);
            if (d >= GX && dw) dma_w(kw, pw, d - GX);
          }
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(Ac[i]), "v"(Bc[j]));
#pragma unroll
        for (int r = 0; r < DR; ++r)
          if (k == 1 + r * (MF / 2) / DR && rd) {
            if (r < FP)
              asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(An[r]) : "v"(la), "i"(r * 2048));
            else
              asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(Bn[r - FP]) : "v"(lb), "i"((r - FP) * 2048));
          }
      }
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  // prologue: every slot's loads in flight, stage 0 visible, (0, 0) read
  uint32_t kw = (uint32_t)rot * 128u, kx = kw;         // of the next stage to load
#pragma unroll
  for (int u = 0; u <= DW; ++u)
    if (u < n2) {
#pragma unroll
      for (int d = 0; d < GW; ++d) dma_w(kw, u * SUBW, d);
      if (u <= DX) {
#pragma unroll
        for (int d = 0; d < GX; ++d) dma_x(kw, u * SUBX, d);
        kx = kw = next_k(kw);
      } else {
        kx = kw;                                       // DW == DX + 1: x is one stage behind
        kw = next_k(kw);
      }
    }
  clear();
  // wait for stage 0: what may still be under way is what was issued behind it
  auto behind = [](int w, int x) constexpr { return w * GW + x * GX; };
  if (n2 > DW) p4_vmcnt<behind(DW, DX)>();
  else if (DW > 4 && n2 == 5) p4_vmcnt<behind(4, DX < 4 ? DX : 4)>();
  else if (DW > 3 && n2 == 4) p4_vmcnt<behind(3, DX < 3 ? DX : 3)>();
  else if (DW > 2 && n2 == 3) p4_vmcnt<behind(2, DX < 2 ? DX : 2)>();
  else if (DW > 1 && n2 == 2) p4_vmcnt<behind(1, 1)>();
  else p4_vmcnt<0>();
  p4_sync();
  rd2(A0, B0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  phase(A0, B0, 0, 0, 1, A1, B1, 0, 0, 0, 0, yes, no, no);   // P_0: (0, 0) on R0, read (0, 1)
  squares(B0, wr == 0);
  int lw = SUBW, lx = SUBX, pw = 0, px = 0;            // byte offsets of the slots of stage s2, and of the one before it
  // stage s2, of which `left` follow (DW stands for DW and more)
  auto stage = [&](auto leftc) {
    constexpr int left = decltype(leftc)::value;
    constexpr int ow = left < DW - 1 ? left : DW - 1, ox = left < DX - 1 ? left : DX - 1;
    constexpr std::integral_constant<bool, (left >= DX)> dx{};
    constexpr std::integral_constant<bool, (left >= DW)> dw{};
    p4_vmcnt<behind(ow, ox)>();                        // stage s2 landed (this wave's DMA), later ones may be under way
    p4_sync();                                         // ... for every wave; (s2 - 1, 1) reads retired
    __builtin_amdgcn_sched_barrier(0);
    phase(A1, B1, lw, lx, 0, A0, B0, kw, pw, kx, px, yes, dx, dw);   // A: (s2 - 1, 1) on R1, read (s2, 0), DMA
    squares(B1, wr == 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    phase(A0, B0, lw, lx, 1, A1, B1, 0, 0, 0, 0, yes, no, no);       // P: (s2, 0) on R0, read (s2, 1)
    squares(B0, wr == 0);
    pw = lw;
    px = lx;
    lw = lw == DW * SUBW ? 0 : lw + SUBW;
    lx = DX == 1 ? SUBX - lx : lx == DX * SUBX ? 0 : lx + SUBX;
    if constexpr (DW == DX) {
      kx = kw = next_k(kw);
    } else {
      kx = kw;
      kw = next_k(kw);
    }
  };
  for (int s2 = 1; s2 < n2 - DW; ++s2) stage(std::integral_constant<int, DW>{});
  auto tail = [&](auto leftc) {
    constexpr int left = decltype(leftc)::value;
    if constexpr (left < DW)
      if (n2 - 1 > left) stage(leftc);
  };
  static_assert(DW <= 5, "tail stages");
  tail(std::integral_constant<int, 4>{});
  tail(std::integral_constant<int, 3>{});
  tail(std::integral_constant<int, 2>{});
  tail(std::integral_constant<int, 1>{});
  tail(std::integral_constant<int, 0>{});
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  phase(A1, B1, 0, 0, 0, A0, B0, 0, 0, 0, 0, no, no, no);   // the last sub-step, (n2 - 1, 1), on R1
  squares(B1, wr == 1);
  p4_vmcnt<0>();
  {   // ... and the last MFMAs' results wait out the MFMA latency before the epilogue reads them:
    // the padding, then one tied empty asm per accumulator (so no read is hoisted above the padding)
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
      for (int j = 0; j < FQ; ++j) asm volatile("" : "+a"(acc[i][j]));
  }

  if constexpr (RMS) {
    __syncthreads();                                     // rss lies in the last stage's memory
#pragma unroll
    for (int f = 0; f < FQ; ++f) {
      ss[f] = lane_sum<16>(ss[f]);
      ss[f] = lane_sum<32>(ss[f]);
    }
    if (g == 0) {
#pragma unroll
      for (int f = 0; f < FQ; ++f) rss[wr * BQ + wc * (BQ / 2) + f * 16 + li] = ss[f];
    }
    __syncthreads();
    if (tid < BQ) rss[tid] += rss[BQ + tid];
    __syncthreads();
  }

  // ---- split-K: raw partial sums into this slice's slab (natural [M][W rows] layout)
  if (a.splits > 1) {
    float* sl = a.slab + (size_t)slice * a.M * a.wrows;
#pragma unroll
    for (int j = 0; j < FQ; ++j) {
      const int m = mt * BQ + wc * (BQ / 2) + j * 16 + li;
      if (m >= a.M) continue;
#pragma unroll
      for (int i = 0; i < FP; ++i) {
        int r0;
        if constexpr (MIX) {
          const int f = nt * (BP / 2) + wr * (BP / 4) + i * 8 + 2 * g;
          if (f >= a.N_out) continue;
          float* row = sl + (size_t)m * a.wrows;
          *reinterpret_cast<p4_f32x2*>(row + f) = p4_f32x2{acc[i][j][0], acc[i][j][1]};
          *reinterpret_cast<p4_f32x2*>(row + a.half_rows + f) = p4_f32x2{acc[i][j][2], acc[i][j][3]};
          continue;
        } else if constexpr (PAIR) {
          const int hf = i / (FP / 2), f = nt * (BP / 2) + wr * (BP / 4) + (i % (FP / 2)) * 16 + 4 * g;
          if (f >= a.N_out) continue;
          r0 = hf ? a.half_rows + f : f;
        } else {
          r0 = nt * BP + wr * (BP / 2) + i * 16 + 4 * g;
          if (r0 >= a.N_out) continue;
        }
        *reinterpret_cast<f32x4*>(sl + (size_t)m * a.wrows + r0) = acc[i][j];
      }
    }
    if (RMS && tid < BQ && mt * BQ + tid < a.M)
      a.slab[(size_t)a.splits * a.M * a.wrows + (size_t)slice * a.M + mt * BQ + tid] = rss[tid];
    return;
  }

  // ---- epilogue: lane holds out[token li of fragment j][features 4 g .. 4 g + 3 of fragment i] (MIX: 2 g, 2 g + 1 of 8)
  constexpr int OF = PAIR && !MIX ? FP / 2 : FP;     // fragments of output features
  constexpr int FF = MIX ? 8 : 16, LF = FF / 4;      // features of one, and of a lane in it
  auto rms = [&](int mloc) -> float {
    if constexpr (RMS) return rsqrtf(rss[mloc] / (float)a.K + a.eps);
    else if constexpr (NORM == P4_SCALED) return a.scale[min(m0 + mloc, m_end - 1)];
    else return 1.f;
  };
  // the LF features of fragments (i, j): the sums with their scale, bias and activation
  auto value = [&](int i, int j, int n0, float sx, float* v) {
    if constexpr (EPI == P4_GLU) {
      f32x4 bg = {0.f, 0.f, 0.f, 0.f}, bu = bg;
      if (a.bias != nullptr) {
        if constexpr (MIX) {                         // (n0 and N_out are even)
          const uint32_t p = *reinterpret_cast<const uint32_t*>(a.bias + n0);
          const uint32_t q = *reinterpret_cast<const uint32_t*>(a.bias + a.half_rows + n0);
          bg = f32x4{lo_bf(p), hi_bf(p), 0.f, 0.f};
          bu = f32x4{lo_bf(q), hi_bf(q), 0.f, 0.f};
        } else {
          bg = ldf4(a.bias + n0);
          bu = ldf4(a.bias + a.half_rows + n0);
        }
      }
#pragma unroll
      for (int e = 0; e < LF; ++e) {
        const float up = MIX ? acc[i][j][2 + e] : acc[FP / 2 + i][j][e];
        v[e] = epi_pair<KIND>(acc[i][j][e] + bg[e], up + bu[e], limit, a.alpha);
      }
    } else if constexpr (EPI == P4_SWIGLU) {
#pragma unroll
      for (int e = 0; e < LF; ++e) {
        const float up = MIX ? acc[i][j][2 + e] : acc[FP / 2 + i][j][e];
        v[e] = p4_silu(acc[i][j][e] * sx) * (up * sx);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] * sx;
      if constexpr (EPI == P4_ACT) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.f ? v[e] * v[e] : 0.f;      // kind 7
      }
    }
  };
  const int nw = nt * (2 * FF * OF) + wr * (FF * OF);    // the wave's first feature
  if constexpr (EPI != P4_F32) {
    if (a.wide) {
      // bf16 rows through LDS: the wave's 16 FQ tokens x FF OF features in the ring's memory (16-byte chunk c of a row in slot
      // c ^ row), then 16 bytes a lane in row order -- whole 64 - 256-byte runs of a row a store, where the registers' order
      // gives 32-byte pieces of 16 rows
      constexpr int CH = FF * OF / 8, NC = CH <= 2 ? 2 : CH <= 4 ? 4 : CH <= 8 ? 8 : 16, ROW = 16 * NC, SH = NC == 4 ? 1 : 0;   // CH of NC chunks
      static_assert(FF * OF % 8 == 0 && 4 * 16 * FQ * ROW <= RING, "the tile's rows fit the ring");
      __syncthreads();                               // every wave has read its last fragments
      char* mine = lds + wid * (16 * FQ * ROW);
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        const int row = j * 16 + li, sw = (row >> SH) & (NC - 1);
        const float sx = rms(wc * (BQ / 2) + row);
#pragma unroll
        for (int i = 0; i < OF; ++i) {
          float v[4];
          value(i, j, min(nw + i * FF + LF * g, a.N_out - LF), sx, v);
          if constexpr (MIX)
            *reinterpret_cast<uint32_t*>(mine + row * ROW + ((i ^ sw) << 4) + g * 4) = pack_bf2(v[0], v[1]);
          else
            *reinterpret_cast<p4_u32x2*>(mine + row * ROW + (((2 * i + (g >> 1)) ^ sw) << 4) + (g & 1) * 8) =
                p4_u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
        }
      }
      asm volatile("" ::: "memory");                 // the wave's own LDS operations run in order
      __builtin_amdgcn_wave_barrier();
      const int c = lane % NC;
#pragma unroll
      for (int p = 0; p < (16 * FQ * NC + 63) / 64; ++p) {
        const int row = p * (64 / NC) + lane / NC, m = m0 + wc * (BQ / 2) + row, n0 = nw + c * 8;
        if (16 * FQ * NC < 64 && row >= 16 * FQ) break;
        const u32x4 o = *reinterpret_cast<const u32x4*>(mine + row * ROW + ((c ^ ((row >> SH) & (NC - 1))) << 4));
        if (m < m_end && n0 < a.N_out && (CH == NC || c < CH))
          *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(a.out) + (size_t)m * a.N_out + n0) = o;
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < FQ; ++j) {
    const int mloc = wc * (BQ / 2) + j * 16 + li;
    const int m = m0 + mloc;
    if (m >= m_end) continue;
    const float sx = rms(mloc);
#pragma unroll
    for (int i = 0; i < OF; ++i) {
      const int n0 = nw + i * FF + LF * g;
      if (n0 >= a.N_out) continue;
      float v[4];
      value(i, j, n0, sx, v);
      if constexpr (MIX) {
        *reinterpret_cast<uint32_t*>(reinterpret_cast<bf16_t*>(a.out) + (size_t)m * a.N_out + n0) = pack_bf2(v[0], v[1]);
      } else if constexpr (EPI == P4_F32) {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + (size_t)m * a.N_out + n0) =
            f32x4{v[0], v[1], v[2], v[3]};
      } else {
        if constexpr (EPI == P4_BF16) {
          if (a.res != nullptr) {
            const p4_u32x2 rr = *reinterpret_cast<const p4_u32x2*>(a.res + (size_t)m * a.N_out + n0);
            v[0] += lo_bf(rr[0]);
            v[1] += hi_bf(rr[0]);
            v[2] += lo_bf(rr[1]);
            v[3] += hi_bf(rr[1]);
          }
        }
        const p4_u32x2 o = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
        *reinterpret_cast<p4_u32x2*>(reinterpret_cast<bf16_t*>(a.out) + (size_t)m * a.N_out + n0) = o;
      }
    }
  }
#endif
}

struct P4Cfg {
  int fp, fq, dw, dx;
};
// tile configurations: BP = 32 FP weight rows x BQ = 32 FQ tokens, 4 waves of (BP / 2) x (BQ / 2)
constexpr P4Cfg kP4Cfgs[] = {
    {8, 8, 2, 1},   // 0: 256 x 256
    {8, 4, 2, 1},   // 1: 256 x 128
    {4, 8, 2, 1},   // 2: 128 x 256
    {4, 4, 2, 1},   // 3: 128 x 128
    {8, 8, 2, 1},   // 4: as 0 (saved plans name it)
    {4, 2, 2, 1},   // 5: 128 x 64
    {2, 2, 4, 4},   // 6: 64 x 64
    {7, 8, 2, 1},   // 7: 224 x 256
    {8, 6, 2, 1},   // 8: 256 x 192
    // a product takes whole rounds of tiles over the CUs, so the menu has tiles for what lies between: of 222 products of 161 - 2100 rows
    // (20 weight shapes, weights cold) the rule's picks take 3.5 % less time on average than the best of those above by its own: 1534 x 2048 x
    // 2048 20.1 -> 16.5 us (128 x 96), 2048 x 3072 x 1536 23.5 -> 21.0 (192 x 128), 1300 x 10240 x 8192 189 -> 155 (256 x 224), grouped 4600 rows
    // of 9 x 2 x 2048 x 2048 89 -> 85 (192 x 224)
    {4, 3, 2, 1},   // 9: 128 x 96
    {6, 3, 2, 1},   // 10: 192 x 96
    {6, 4, 2, 1},   // 11: 192 x 128
    {4, 6, 2, 1},   // 12: 128 x 192
    {6, 6, 2, 1},   // 13: 192 x 192
    {7, 6, 2, 1},   // 14: 224 x 192
    {6, 7, 2, 1},   // 15: 192 x 224 (ungrouped for tuned plans alone: ops/__init__.py has no figures for it off the table)
    {7, 7, 2, 1},   // 16: 224 x 224
    {8, 7, 2, 1},   // 17: 256 x 224
};
constexpr int kP4NumCfgs = sizeof(kP4Cfgs) / sizeof(kP4Cfgs[0]);
// tiles of 32 tokens, of the grouped form only (configurations kP4NumCfgs and up), two workgroups on a CU: groups of a few rows are a
// stream of weights, at which the CUs are equally busy only if the tiles fill a whole number of rounds, so several widths.  Which one:
// ops/seqmix.py _grouped_few.  us, tiles of 64 and 128 rows / these, 8 groups and a common one, weights from memory: gated 2 x 2048 x 2048, 32
// tokens 36.1 / 31.3 (160 x 32), 8 27.6 / 26.6; 2048 x 2048, 32 21.8 / 18.1 (96 x 32); 4096 x 3584, 16 55.8 / 49.2.
constexpr P4Cfg kP4Few[] = {
    {2, 1, 4, 4},   // 18: 64 x 32
    {3, 1, 3, 3},   // 19: 96 x 32
    {4, 1, 3, 3},   // 20: 128 x 32
    {5, 1, 2, 2},   // 21: 160 x 32
};
constexpr int kP4Grouped = kP4NumCfgs + sizeof(kP4Few) / sizeof(kP4Few[0]);
constexpr P4Cfg p4_tile(int c) { return c < kP4NumCfgs ? kP4Cfgs[c] : kP4Few[c - kP4NumCfgs]; }
// the walks of P4Args::spread and fine, and what goes with them
inline void p4_walk(P4Args& a, int cfg) {
  const P4Cfg t = p4_tile(cfg);
  if (a.K <= 2048 && (t.fq == 1 || (t.fp <= 4 && t.fq <= 4))) {
    a.spread = 1;
    a.fine = 4;
  } else if (a.K >= 16384 && a.m_tiles <= 8 && a.groups == 0) {
    a.spread = 1;
    if (a.group_m < a.m_tiles) a.group_m = a.m_tiles;
  }
}

template <int C, int EPI, int NORM>
int p4_launch(const P4Args& a, hipStream_t s) {
  hipLaunchKernelGGL((pgemm4_kernel<kP4Cfgs[C].fp, kP4Cfgs[C].fq, kP4Cfgs[C].dw, kP4Cfgs[C].dx, EPI, NORM>), dim3(a.nwg),
                     dim3(256), 0, s, a);
  return (int)hipGetLastError();
}
// row scales that are given: the tiles of large products only
constexpr bool p4_scaled(int cfg) { return kP4Cfgs[cfg].fp * kP4Cfgs[cfg].fq >= 32; }
template <int C>
int p4_epi(const P4Args& a, int epi, int norm, hipStream_t s) {
  if (norm == P4_SCALED) {
    if constexpr (p4_scaled(C)) {
      if (epi == P4_BF16) return p4_launch<C, P4_BF16, P4_SCALED>(a, s);
      if (epi == P4_SWIGLU) return p4_launch<C, P4_SWIGLU, P4_SCALED>(a, s);
    }
  } else if (norm == P4_RMS) {
    switch (epi) {
      case P4_BF16: return p4_launch<C, P4_BF16, P4_RMS>(a, s);
      case P4_F32: return p4_launch<C, P4_F32, P4_RMS>(a, s);
      case P4_SWIGLU: return p4_launch<C, P4_SWIGLU, P4_RMS>(a, s);
    }
  } else {
    switch (epi) {
      case P4_BF16: return p4_launch<C, P4_BF16, P4_PLAIN>(a, s);
      case P4_F32: return p4_launch<C, P4_F32, P4_PLAIN>(a, s);
      case P4_SWIGLU: return p4_launch<C, P4_SWIGLU, P4_PLAIN>(a, s);
    }
  }
  return -2;
}
template <int C, int END>
int p4_cfg(const P4Args& a, int cfg, int epi, int rms, hipStream_t s) {
  if constexpr (C < END) {
    if (cfg == C) return p4_epi<C>(a, epi, rms, s);
    return p4_cfg<C + 1, END>(a, cfg, epi, rms, s);
  } else {
    return -4;
  }
}

// The forms with an activation (gated kinds 0, 1, 5; elementwise 7) and the grouped ones.
template <int C, int EPI, bool GRP, int KIND>
int p4_act_launch(const P4Args& a, hipStream_t s) {
  constexpr P4Cfg T = p4_tile(C);
  hipLaunchKernelGGL((pgemm4_kernel<T.fp, T.fq, T.dw, T.dx, EPI, P4_PLAIN, GRP, KIND>), dim3(a.nwg), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}
template <int C, bool GRP>
int p4_act_kind(const P4Args& a, int kind, hipStream_t s) {
  switch (kind) {
    case 0: return p4_act_launch<C, P4_GLU, GRP, 0>(a, s);
    case 1: return p4_act_launch<C, P4_GLU, GRP, 1>(a, s);
    case 5: return p4_act_launch<C, P4_GLU, GRP, 5>(a, s);
    case 7:
      if constexpr (!GRP) return p4_act_launch<C, P4_ACT, false, 7>(a, s);
      break;
    case -1:
      if constexpr (GRP) return p4_act_launch<C, P4_BF16, true, -1>(a, s);
      break;
  }
  return -1;
}
// the grouped form is built on the tiles that ops/seqmix.py's rules take
constexpr bool p4_grouped(int cfg) { return cfg != 9 && cfg != 14; }
template <bool GRP, int C, int END>
int p4_act_cfg(const P4Args& a, int cfg, int kind, hipStream_t s) {
  if constexpr (C < END) {
    if constexpr (!GRP || p4_grouped(C)) {
      if (cfg == C) return p4_act_kind<C, GRP>(a, kind, s);
    }
    return p4_act_cfg<GRP, C + 1, END>(a, cfg, kind, s);
  } else {
    return -4;
  }
}

// configurations [P4_TILES, P4_WIDE) in pgemm4_tiles.hip, [P4_WIDE, kP4NumCfgs) and those of 32 tokens in pgemm4_wide.hip
constexpr int P4_TILES = 9, P4_WIDE = 14;
int p4_tiles(const P4Args& a, int cfg, int epi, int norm, hipStream_t s);
int p4_tiles_act(const P4Args& a, int cfg, int kind, bool grouped, hipStream_t s);
int p4_wide(const P4Args& a, int cfg, int epi, int norm, hipStream_t s);
int p4_wide_act(const P4Args& a, int cfg, int kind, bool grouped, hipStream_t s);

}  // namespace k8sllm
