// The kernels of sgemv.hip (its notes are there), and of the MFMA form also its launch, for sgemv_act.hip too.
#pragma once

#include <atomic>
#include <cstdlib>

#include "act.h"
#include "common.h"

namespace k8sllm {

namespace {

constexpr int SG_BAND = 64;   // most output rows per workgroup band (LDS partials: KW x 2*BAND x MT floats)
// GLU, ELEM: an activation of act.h, gated (W as for SWIGLU) or elementwise, bf16 output (sgemv_act.hip)
enum SgEpi { SG_BF16 = 0, SG_F32 = 1, SG_SWIGLU = 2, SG_GLU = 3, SG_ELEM = 4 };
constexpr bool sg_paired(int epi) { return epi == SG_SWIGLU || epi == SG_GLU; }

__device__ __forceinline__ float sg_dot2(uint32_t w, uint32_t x, float acc) {
  bf16x2 a, b;
  __builtin_memcpy(&a, &w, 4);
  __builtin_memcpy(&b, &x, 4);
  return __builtin_amdgcn_fdot2_f32_bf16(a, b, acc, false);
}
__device__ __forceinline__ float sg_dot8(const u32x4& w, const u32x4& x, float acc) {
  acc = sg_dot2(w.x, x.x, acc);
  acc = sg_dot2(w.y, x.y, acc);
  acc = sg_dot2(w.z, x.z, acc);
  return sg_dot2(w.w, x.w, acc);
}
// Halving butterfly over the 64 lanes for CNT values per lane: at xor offset O a lane keeps half of its values
// (the lower half if bit O of its lane id is clear) and adds the partner's copy of that half.  Once one value is
// left, the remaining offsets are plain xor sums.  Afterwards value index (lane >> (6 - log2 V)) & (V - 1) of the
// ORIGINAL V values is the wave total in v[0] of every lane (all lanes of a group agree).
template <int O>
__device__ __forceinline__ float sg_keep(float a, float b, int lane) {   // lanes without bit O: a, the others: b, of both lanes
  if constexpr (O >= 16) {
    float x, y;
    lane_swap<O>(a, b, x, y);
    return x + y;
  } else {
    const bool up = (lane & O) != 0;
    return (up ? b : a) + lane_xor<O>(up ? a : b);
  }
}
template <int CNT, int O>
__device__ __forceinline__ void sg_halve(float* v, int lane) {
  if constexpr (O >= 1) {
    if constexpr (CNT > 1) {
#pragma unroll
      for (int i = 0; i < CNT / 2; ++i) v[i] = sg_keep<O>(v[i], v[i + CNT / 2], lane);
      sg_halve<CNT / 2, O / 2>(v, lane);
    } else {
      v[0] = lane_sum<O>(v[0]);
      sg_halve<1, O / 2>(v, lane);
    }
  }
}
template <int V>
constexpr int sg_log2() { return V <= 1 ? 0 : 1 + sg_log2<V / 2>(); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t sg_rsrc(const void* p, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)min(bytes, 0x7fffffffLL), 0x00020000);
}

}  // namespace

// MT: rows of x the kernel is built for (4 or 8; the first M are live).  KPW: k elements per wave slice.  KW: waves
// per workgroup that split K.  NORM: 1/rms of each x row (gamma folded into W) from the x registers (needs the
// workgroup to cover all of K: G == 1).  RES: out = res + acc (res may alias out).  FP8: W is e4m3 with per-row
// fp32 scales wscale.
template <int MT, int KPW, int KW, int EPI, bool NORM, bool RES, bool FP8>
__global__ void __launch_bounds__(256) sgemv_kernel(void* __restrict__ out, float* __restrict__ part,
                                                     const bf16_t* __restrict__ x, const void* __restrict__ W,
                                                     const float* __restrict__ wscale, const bf16_t* res, int M,
                                                     int N, int K, float eps, int half_rows, int band_rows) {
  constexpr int EPC = FP8 ? 16 : 8;            // elements per 16-byte weight chunk
  constexpr int CPL = KPW / (64 * EPC);         // chunks per lane
  constexpr int XV = FP8 ? 2 : 1;               // x vectors (u32x4) per chunk and row
  constexpr int NR = (EPI == SG_SWIGLU) ? 1 : 2;   // output rows per step
  constexpr int NRT = (EPI == SG_SWIGLU) ? 2 : NR; // weight rows per step (gate and up)
  constexpr int V = NRT * MT;                   // partial sums per lane per step
  constexpr int LV = sg_log2<V>();
  constexpr int RGN = 4 / KW;                   // row groups
  constexpr int WB = FP8 ? 1 : 2;               // weight bytes
  static_assert(CPL >= 1 && V <= 64 && (V & (V - 1)) == 0, "bad sgemv configuration");
  __shared__ float red[KW][NRT * SG_BAND][MT];
  __shared__ float ssr[KW][MT];

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int kw = wid % KW, rg = wid / KW;
  const int g = blockIdx.y;
  const int nch = K / EPC;                      // chunks per weight row
  const int cb = (g * KW + kw) * (64 * CPL);    // this wave's first chunk
  const bool active = cb < nch;
  const int b0 = blockIdx.x * band_rows;           // band_rows <= SG_BAND (the LDS partials' capacity)
  const int band = min(band_rows, N - b0);
  const int nsets = (band + NR - 1) / NR;
  const char* Wb = reinterpret_cast<const char*>(W);
  const long long row_bytes = (long long)K * WB;

  // ---- x slice into registers (rows >= M and chunks past K read 0 through the buffer bounds)
  u32x4 xr[CPL][MT][XV];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    // one buffer resource per x row, bounded by the row (0 bytes for rows >= M): chunks past K and dead rows load
    // 0 without a branch (a per-load select made the compiler wait for each load separately)
    const auto xs = sg_rsrc(x + (size_t)min(m, M - 1) * K, m < M ? (long long)K * 2 : 0);
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int c = cb + 64 * j + lane;
#pragma unroll
      for (int v = 0; v < XV; ++v) xr[j][m][v] = __builtin_amdgcn_raw_buffer_load_b128(xs, c * EPC * 2 + 16 * v, 0, 0);
    }
  }

  // one row set: NRT weight rows x CPL chunks per lane (clamped to the row: x is 0 there)
  auto load_set = [&](u32x4 (&w)[CPL][NRT], int q) {
#pragma unroll
    for (int r = 0; r < NRT; ++r) {
      const int rl = (EPI == SG_SWIGLU) ? q : q * NR + r;
      const int n = min(b0 + min(rl, band - 1), N - 1) + ((EPI == SG_SWIGLU && r == 1) ? half_rows : 0);
      const u32x4* row = reinterpret_cast<const u32x4*>(Wb + (long long)n * row_bytes);
#pragma unroll
      for (int j = 0; j < CPL; ++j) w[j][r] = __builtin_nontemporal_load(row + min(cb + 64 * j + lane, nch - 1));
    }
  };
  auto consume = [&](const u32x4 (&w)[CPL][NRT], int q) {
    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j)
#pragma unroll
      for (int r = 0; r < NRT; ++r) {
        if constexpr (FP8) {
          // the 16 e4m3 weights become 8 exact bf16 pairs ONCE, then meet every x row (not once per row)
          bf16x2 wp[8];
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            wp[2 * d] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[j][r][d], 1.0f, false);
            wp[2 * d + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[j][r][d], 1.0f, true);
          }
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            float a = acc[r * MT + m];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const uint32_t xw = e < 4 ? xr[j][m][0][e] : xr[j][m][1][e - 4];
              bf16x2 xb;
              __builtin_memcpy(&xb, &xw, 4);
              a = __builtin_amdgcn_fdot2_f32_bf16(wp[e], xb, a, false);
            }
            acc[r * MT + m] = a;
          }
        } else {
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[r * MT + m] = sg_dot8(w[j][r], xr[j][m][0], acc[r * MT + m]);
        }
      }
    sg_halve<V, 32>(acc, lane);
    if ((lane & ((1 << (6 - LV)) - 1)) == 0) {
      const int idx = (lane >> (6 - LV)) & (V - 1);
      const int r = idx / MT, m = idx % MT;
      const int rl = (EPI == SG_SWIGLU) ? q + r * SG_BAND : q * NR + r;
      red[kw][rl][m] = acc[0];
    }
  };

  // the first row set's weights go out right behind the x loads, unconditionally (rows and chunks are clamped, so a
  // wave with no set or no slice reads valid bytes it ignores): a branch here let the compiler sink them below the
  // norm prologue, which then waited for every x load before a single weight byte was requested
  u32x4 wa[CPL][NRT], wb[CPL][NRT];
  int q = rg;
  asm volatile("" ::: "memory");   // every x load is issued before the first weight load (in-order retirement)
  load_set(wa, q);
  asm volatile("" ::: "memory");
  // and the x registers become opaque only here, so nothing that reads them (the norm's sum of squares) can be
  // scheduled above the weight loads: its wait is then for the x loads only (counted: the weights stay in flight)
  if constexpr (NORM) {
#pragma unroll
    for (int j = 0; j < CPL; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int v = 0; v < XV; ++v) asm volatile("" : "+v"(xr[j][m][v]));
  }

  if constexpr (NORM) {   // sum of squares of each live x row over this wave's slice (the weights are in flight)
    float ss[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < CPL; ++j)
#pragma unroll
        for (int v = 0; v < XV; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float lo = lo_bf(xr[j][m][v][e]), hi = hi_bf(xr[j][m][v][e]);
            s += lo * lo + hi * hi;
          }
      ss[m] = s;
    }
    constexpr int LM = sg_log2<MT>();
    sg_halve<MT, 32>(ss, lane);
    if (rg == 0 && (lane & ((1 << (6 - LM)) - 1)) == 0) ssr[kw][(lane >> (6 - LM)) & (MT - 1)] = ss[0];
  }

  if (active) {
    for (; q < nsets; q += 2 * RGN) {
      if (q + RGN < nsets) load_set(wb, q + RGN);
      consume(wa, q);
      if (q + RGN >= nsets) break;
      if (q + 2 * RGN < nsets) load_set(wa, q + 2 * RGN);
      consume(wb, q + RGN);
    }
  } else {   // a slice past the end of K (the last k-group of a ragged split): contributes zeros
    for (int i = lane; i < NRT * SG_BAND * MT; i += 64) (&red[kw][0][0])[i] = 0.f;
  }
  __syncthreads();

  // ---- combine the k-slices (fixed order), scale, epilogue
  const int G = gridDim.y;
  for (int t = threadIdx.x; t < band * MT; t += 256) {
    const int m = t / band, rl = t - m * band;
    if (m >= M) break;
    const int n = b0 + rl;
    float a = 0.f, u = 0.f;
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      a += red[k][rl][m];
      if (EPI == SG_SWIGLU) u += red[k][SG_BAND + rl][m];
    }
    if constexpr (NORM) {
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < KW; ++k) s += ssr[k][m];
      const float inv = rsqrtf(s / (float)K + eps);
      a *= inv;
      u *= inv;
    }
    if constexpr (FP8) {
      a *= wscale[n];
      if (EPI == SG_SWIGLU) u *= wscale[n + half_rows];
    }
    if (G > 1) {   // partial slab of this k-group; sgemv_finalize_kernel applies the epilogue
      const int wrows = (EPI == SG_SWIGLU) ? 2 * N : N;
      float* slab = part + ((size_t)g * M + m) * wrows;
      slab[n] = a;
      if (EPI == SG_SWIGLU) slab[N + n] = u;
      continue;
    }
    if constexpr (EPI == SG_F32) {
      reinterpret_cast<float*>(out)[(size_t)m * N + n] = a;
    } else if constexpr (EPI == SG_SWIGLU) {
      reinterpret_cast<bf16_t*>(out)[(size_t)m * N + n] = f2bf(a / (1.f + __expf(-a)) * u);
    } else {
      if constexpr (RES) a += bf2f(res[(size_t)m * N + n]);
      reinterpret_cast<bf16_t*>(out)[(size_t)m * N + n] = f2bf(a);
    }
  }
}

// 5..16 decode rows on the MATRIX cores.  At 8 rows the v_dot2 form above issues 32 VALU dot2 per 16 weight bytes
// (fp8: 72 with the conversions): VALU-bound at ~5 TB/s (fp8 ~3 TB/s), and it cannot hold 16 rows of x.  Here the
// products run on v_mfma_f32_4x4x4bf16_1k -- 16 independent 4x4x4 blocks, lane 4b + i holding row i of block b
// (A: weights, items = 4 k; B: x, column j = lane & 3; D: item i of lane 4b + j = D[i][j]; checked on the chip by
// tools/experiments/mfma4_layout.hip) -- so the VALU is free and the kernel is a pure weight stream again:
//  * one 16-byte-per-lane load covers 4 weight rows x 256 contiguous bytes (lane l: row l & 3, chunk l >> 2): the
//    16 blocks are 16 consecutive chunks of the same 4 rows, each chunk two (bf16) or four (fp8) k-quads.  That
//    access shape streams at ~6.2 TB/s where the 16x16x32 MFMA's A operand (16 rows x 64 B per load) manages ~5.0
//    (tools/experiments/ldpat.hip, profiles/sgemv_load_patterns_r4.txt);
//  * x lives in registers for the whole launch (B operand: x row 4 xg + (l & 3), the same chunks), MT / 4 groups
//    of 4 rows; fp8 weights become bf16 k-quads with v_cvt_scalef32_pk_bf16_fp8 (x stays bf16, the row scale
//    lands in the epilogue);
//  * 512 threads = 8 waves, ALL splitting the workgroup's k range (jw steps of 16 chunks each); the workgroup
//    walks its band in quads of 4 rows (SwiGLU: gate quads then up quads), register sets of 4 loads (4 KiB per
//    wave) double-buffered -- the shallow queue streams best (the probe: 4-8 KiB per wave beats 16-32 KiB);
//  * at the end of a quad the 16 blocks' partial products are summed by a halving butterfly (4 x MT / 4 values per
//    lane, offsets 32..4) and parked in LDS; after the band the 8 k-slices are summed in a fixed order
//    (deterministic) and the norm / scale / epilogue applied as in the v_dot2 form;
//  * band sized for about one workgroup per CU and k-group; steps past a wave's slice and rows past the band are
//    out of range of the load's buffer (0, no traffic) instead of branches, so every wait is a counted one.
constexpr int SM_KW = 8;   // waves per workgroup

template <int CNT, int O>
__device__ __forceinline__ void sm_halve(float* v, int lane) {   // sg_halve that stops at offset 4 (j = lane & 3)
  if constexpr (O >= 4) {
    if constexpr (CNT > 1) {
#pragma unroll
      for (int i = 0; i < CNT / 2; ++i) v[i] = sg_keep<O>(v[i], v[i + CNT / 2], lane);
      sm_halve<CNT / 2, O / 2>(v, lane);
    } else {
      v[0] = lane_sum<O>(v[0]);
      sm_halve<1, O / 2>(v, lane);
    }
  }
}

template <int EPI, bool RES>
__device__ __forceinline__ void sm_store(void* out, size_t o, float a, float u, float rv, const EpiAct& act) {
  if constexpr (EPI == SG_F32) {
    reinterpret_cast<float*>(out)[o] = a;
  } else if constexpr (EPI == SG_SWIGLU) {
    reinterpret_cast<bf16_t*>(out)[o] = f2bf(a / (1.f + __expf(-a)) * u);
  } else if constexpr (EPI == SG_GLU) {
    reinterpret_cast<bf16_t*>(out)[o] = f2bf(epi_gated(a, u, act));
  } else if constexpr (EPI == SG_ELEM) {
    reinterpret_cast<bf16_t*>(out)[o] = f2bf(epi_elem(a, act));
  } else {
    if constexpr (RES) a += rv;
    reinterpret_cast<bf16_t*>(out)[o] = f2bf(a);
  }
}

// Tickets of the in-kernel k-group reduction: zero at load, each range returned to zero by the last workgroup of
// every launch that used it.  Launches draw ranges of SM_TICKET_RANGE in rotation, so kernels that overlap on
// different streams do not share counters.
constexpr int SM_TICKET_RANGE = 256, SM_TICKET_RANGES = 256;
__device__ unsigned sm_tickets[SM_TICKET_RANGE * SM_TICKET_RANGES];

// Products of a decode step's few rows (stream_gemv.hip).  Of a normed fp32 stream: ROWS 1 adds to the stream and leaves what the next product's norm needs, ROWS
// 2 reads that: the norm is a factor of each row, which a product's sums can take as well as its input.  ROWS 3: several inputs of M
// rows one after the other, `count` rows of W for each and the rest, past n1, for the last, through tanh to out2.
struct SmRows {
  const float* x;          // 1: y = x + mult * product -> y (another buffer), h = bf16(y (offset + nw)), and of every workgroup's
  float* y;                //    columns the rows' sums of y^2 -> sums[m][blockIdx.x]
  bf16_t* h;
  const bf16_t* nw;
  float* sums;
  const float* sums_in;    // 2: [M][count]; the product times gain / sqrt(sum / K + eps)
  bf16_t* out2;            //    columns from n1 on (n1 = N: none), rows of N - n1; the others: rows of n1
  int count, n1;
  float mult, offset;
};
constexpr int SM_SUMS = 256;   // most workgroups that leave sums of a row

template <int MT, int JT, int EPI, bool NORM, bool RES, bool FP8, int ROWS = 0>
__global__ void __launch_bounds__(512) smfma_kernel(void* __restrict__ out, float* __restrict__ part,
                                                     const bf16_t* __restrict__ x, const void* __restrict__ W,
                                                     const float* __restrict__ wscale, const bf16_t* res, int M,
                                                     int N, int K, float eps, int band_rows, int jw,
                                                     unsigned* tickets, EpiAct act, SmRows rows) {
  constexpr int EPC = FP8 ? 16 : 8;                // k per 16-byte weight chunk
  constexpr int XG = MT / 4;                       // x groups of 4 rows (the B operand's 4 columns)
  constexpr int KQ = EPC / 4;                      // k-quads per chunk
  constexpr int XV = FP8 ? 2 : 1;                  // x u32x4 per chunk and row
  constexpr int Q = 4;                             // loads per register set
  constexpr int QPU = JT >= Q ? 1 : Q / JT;        // quads per set
  constexpr int NSB = JT >= Q ? JT / Q : 1;        // sets per quad block
  constexpr int QMAX = 512 / MT;                   // quads per workgroup (LDS partials: 64 KiB)
  constexpr int V = 4 * XG;                        // partial products per lane and quad
  constexpr int LV = sg_log2<V>();
  constexpr int WB = FP8 ? 1 : 2;
  static_assert((JT & (JT - 1)) == 0 && JT <= 8 && V <= 16, "bad smfma configuration");
  __shared__ float red[SM_KW][QMAX][4][MT];
  __shared__ float ssw[SM_KW][MT];
  __shared__ float sq[ROWS == 1 ? 4 * QMAX * MT : 1];   // ROWS 1: the squares of the workgroup's outputs

  const int tid = threadIdx.x, lane = tid & 63;
  const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);   // (wave-uniform: the step masks below are scalar)
  const int r4 = lane & 3, cb = lane >> 2;         // row in the quad / x row in the group; chunk = block
  const int g = blockIdx.y;
  const int C16 = K / (16 * EPC);                  // steps (16 chunks) per weight row
  const int sb = (g * SM_KW + kw) * jw;            // this wave's first step
  const int jv = max(0, min(jw, C16 - sb));        // its live steps (0: a slice past K)
  const int b0 = blockIdx.x * band_rows;
  const int band = min(band_rows, N - b0);
  const int qg = (band + 3) >> 2;                  // quads of output rows
  const int nq = (sg_paired(EPI)) ? 2 * qg : qg;
  const unsigned row_bytes = (unsigned)K * WB;
  constexpr unsigned OOB = 0x80000000u;            // past every buffer below: the load returns 0, no traffic

  // ---- x -> registers: xr[s][xg] = x[4 xg + r4][chunk 16 (sb + s) + cb]; rows >= M / dead steps read 0
  u32x4 xr[JT][XG][XV];
  {
    // (ROWS 3: all bands past n1 are the last input's, which may have more rows of W than the others)
    const auto xs = sg_rsrc(x + (ROWS == 3 ? (size_t)(min(b0, rows.n1) / rows.count) * M * K : 0), (long long)M * K * 2);
#pragma unroll
    for (int s = 0; s < JT; ++s)
#pragma unroll
      for (int xg = 0; xg < XG; ++xg) {
        const unsigned off =
            s < jv ? (unsigned)(4 * xg + r4) * K * 2 + (unsigned)(16 * (sb + s) + cb) * EPC * 2 : OOB;
#pragma unroll
        for (int v = 0; v < XV; ++v) xr[s][xg][v] = __builtin_amdgcn_raw_buffer_load_b128(xs, off + 16 * v, 0, 0);
      }
  }

  // wave kw's rows' sums, ahead of the weights as the x loads are
  float rs[ROWS == 2 ? MT / SM_KW : 1][SM_SUMS / 64];
  if constexpr (ROWS == 2) {
    const auto ss = sg_rsrc(rows.sums_in, (long long)M * rows.count * 4);
#pragma unroll
    for (int r = 0; r < MT / SM_KW; ++r)
#pragma unroll
      for (int i = 0; i < SM_SUMS / 64; ++i) {
        const int m = kw + SM_KW * r, c = lane + 64 * i;
        rs[r][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                 ss, c < rows.count && m < M ? (unsigned)(m * rows.count + c) * 4 : OOB, 0, 0));
      }
  }

  // the band's weight rows through one buffer per half (gate rows; SwiGLU: up rows)
  const char* Wc = reinterpret_cast<const char*>(W);
  const auto wg = sg_rsrc(Wc + (size_t)b0 * row_bytes, (long long)band * row_bytes);
  const auto wu = sg_rsrc(Wc + ((sg_paired(EPI)) ? (size_t)(N + b0) * row_bytes : 0),
                          (sg_paired(EPI)) ? (long long)band * row_bytes : 0);
  const unsigned lane_off = (unsigned)r4 * row_bytes + (unsigned)(16 * sb + cb) * 16;
  // element e of set i of quad block qb: (quad, step), both compile-time but the block
  auto quad_of = [](int qb, int e) { return qb * QPU + (JT >= Q ? 0 : e / JT); };
  auto step_of = [](int i, int e) { return JT >= Q ? i * Q + e : e % JT; };
  auto load_set = [&](u32x4 (&w)[Q], int qb, int i) {
#pragma unroll
    for (int e = 0; e < Q; ++e) {
      const int quad = quad_of(qb, e), s = step_of(i, e);
      const bool up = sg_paired(EPI) && quad >= qg;
      const unsigned off = s < jv ? (unsigned)(4 * (up ? quad - qg : quad)) * row_bytes + lane_off + 256u * s : OOB;
      w[e] = __builtin_amdgcn_raw_buffer_load_b128(up ? wu : wg, off, 0, 2);   // (aux 2: non-temporal)
    }
  };
  auto consume = [&](const u32x4 (&w)[Q], int i, f32x4 (&acc)[QPU][XG]) {
#pragma unroll
    for (int e = 0; e < Q; ++e) {
      const int qq = JT >= Q ? 0 : e / JT, s = step_of(i, e);
#pragma unroll
      for (int kq = 0; kq < KQ; ++kq) {
        uint32_t a0, a1;
        if constexpr (FP8) {
          a0 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[e][kq], 1.0f, false));
          a1 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[e][kq], 1.0f, true));
        } else {
          a0 = w[e][2 * kq];
          a1 = w[e][2 * kq + 1];
        }
        const bf16x4 a = __builtin_bit_cast(bf16x4, (uint2){a0, a1});
#pragma unroll
        for (int xg = 0; xg < XG; ++xg) {
          const u32x4& xv = xr[s][xg][kq / 2];
          const bf16x4 b = __builtin_bit_cast(bf16x4, (uint2){xv[2 * (kq & 1)], xv[2 * (kq & 1) + 1]});
          acc[qq][xg] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a, b, acc[qq][xg], 0, 0, 0);
        }
      }
    }
  };
  auto park = [&](const f32x4 (&acc)[QPU][XG], int qb) {   // sum the 16 blocks, one lane per (row, x row) to LDS
#pragma unroll
    for (int qq = 0; qq < QPU; ++qq) {
      float v[V];
#pragma unroll
      for (int xg = 0; xg < XG; ++xg)
#pragma unroll
        for (int it = 0; it < 4; ++it) v[xg * 4 + it] = acc[qq][xg][it];
      sm_halve<V, 32>(v, lane);
      const int idx = (lane >> (6 - LV)) & (V - 1);
      if (((lane >> 2) & ((1 << (4 - LV)) - 1)) == 0) red[kw][qb * QPU + qq][idx & 3][4 * (idx >> 2) + r4] = v[0];
    }
  };

  u32x4 wbuf[2][Q];
  asm volatile("" ::: "memory");   // every x load is issued before the first weight load (in-order retirement)
  load_set(wbuf[0], 0, 0);         // (every launched workgroup has >= 1 quad)
  asm volatile("" ::: "memory");
  if constexpr (NORM) {   // sum of squares of each x row over this wave's slice, the first weights in flight
#pragma unroll
    for (int s = 0; s < JT; ++s)
#pragma unroll
      for (int xg = 0; xg < XG; ++xg)
#pragma unroll
        for (int v = 0; v < XV; ++v) asm volatile("" : "+v"(xr[s][xg][v]));
    float ss[XG];
#pragma unroll
    for (int xg = 0; xg < XG; ++xg) {
      float t = 0.f;
#pragma unroll
      for (int s = 0; s < JT; ++s)
#pragma unroll
        for (int v = 0; v < XV; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float lo = lo_bf(xr[s][xg][v][e]), hi = hi_bf(xr[s][xg][v][e]);
            t += lo * lo + hi * hi;
          }
      ss[xg] = lane_sum<32>(lane_sum<16>(lane_sum<8>(lane_sum<4>(t))));
    }
    if (lane < 4) {
#pragma unroll
      for (int xg = 0; xg < XG; ++xg) ssw[kw][4 * xg + lane] = ss[xg];
    }
  }

  if constexpr (ROWS == 2) {
#pragma unroll
    for (int r = 0; r < MT / SM_KW; ++r) {
#pragma unroll
      for (int i = 0; i < SM_SUMS / 64; ++i) asm volatile("" : "+v"(rs[r][i]));
      const float t = wave_sum((rs[r][0] + rs[r][1]) + (rs[r][2] + rs[r][3]));
      if (lane == 0) ssw[0][kw + SM_KW * r] = t;
    }
  }

  // the first epilogue pass's residual and row scales are requested now, behind the first weight set (clamped, so no
  // load sits under a branch): their latency hides under the weight stream instead of ending the kernel
  float pre_res = 0.f, pre_sa = 1.f, pre_su = 1.f;   // (ROWS 1: the stream and the next norm's weight)
  asm volatile("" ::: "memory");
  {
    const int idx = min(tid, band * M - 1);
    const int m = idx / band, n = b0 + idx - m * band;
    if constexpr (RES) pre_res = bf2f(res[(size_t)m * N + n]);
    if constexpr (ROWS == 1) {
      pre_res = rows.x[(size_t)m * N + n];
      pre_sa = bf2f(rows.nw[n]);
    }
    if constexpr (FP8) {
      pre_sa = wscale[n];
      if constexpr (sg_paired(EPI)) pre_su = wscale[N + n];
    }
  }

  // quad blocks two at a time so the register set of every (block, set) pair is a compile-time choice; an odd
  // count runs a phantom block, and the last block prefetches the (out-of-range) block after it: no load sits
  // under a branch, so every wait stays a counted one
  const int nqb = (nq + QPU - 1) / QPU;
  const int nqbp = (nqb + 1) & ~1;   // (host: nqbp * QPU <= QMAX)
  for (int qb = 0; qb < nqbp; qb += 2) {
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const int qbc = qb + tt;
      f32x4 acc[QPU][XG];
#pragma unroll
      for (int qq = 0; qq < QPU; ++qq)
#pragma unroll
        for (int xg = 0; xg < XG; ++xg) acc[qq][xg] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NSB; ++i) {
        const int par = (tt * NSB + i) & 1;
        const int nb = i + 1 < NSB ? qbc : qbc + 1, ni = i + 1 < NSB ? i + 1 : 0;
        if (par) load_set(wbuf[0], nb, ni); else load_set(wbuf[1], nb, ni);
        // the next set's loads go out before this set's MFMAs (and their waits): the barrier keeps the loads
        // above it, the opaque accumulators (and, for fp8, the current set feeding the conversions) the math below
        asm volatile("" ::: "memory");
#pragma unroll
        for (int qq = 0; qq < QPU; ++qq)
#pragma unroll
          for (int xg = 0; xg < XG; ++xg) asm volatile("" : "+v"(acc[qq][xg]));
        if constexpr (FP8) {
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            if (par) asm volatile("" : "+v"(wbuf[1][q])); else asm volatile("" : "+v"(wbuf[0][q]));
          }
        }
        if (par) consume(wbuf[1], i, acc); else consume(wbuf[0], i, acc);
      }
      park(acc, qbc);
    }
  }
  __syncthreads();

  // ---- combine the 8 k-slices (fixed order), scale, epilogue
  const int G = gridDim.y;
  auto store = [&](int idx, int m, int n, float a, float u) {
    const size_t o = (size_t)m * N + n;
    const bool first = idx == tid;
    if constexpr (ROWS == 1) {
      const float y = fmaf(rows.mult, a, first ? pre_res : rows.x[o]);
      rows.y[o] = y;
      rows.h[o] = f2bf(y * (rows.offset + (first ? pre_sa : bf2f(rows.nw[n]))));
      sq[idx] = y * y;
    } else if constexpr (ROWS == 2) {
      const bool second = n >= rows.n1;
      sm_store<EPI, false>(second ? rows.out2 : out, second ? (size_t)m * (N - rows.n1) + (n - rows.n1) : (size_t)m * rows.n1 + n, a,
                           u, 0.f, act);
    } else if constexpr (ROWS == 3) {
      const size_t g = b0 / rows.count;             // (a band lies in one input's rows)
      if (n < rows.n1) reinterpret_cast<bf16_t*>(out)[(g * M + m) * rows.count + (n - g * rows.count)] = f2bf(a);
      else rows.out2[(size_t)m * (N - rows.n1) + (n - rows.n1)] = f2bf(tanhf(a));
    } else {
      sm_store<EPI, RES>(out, o, a, u, RES ? (first ? pre_res : bf2f(res[o])) : 0.f, act);
    }
  };
  auto row_sums = [&]() {   // after the last store
    if constexpr (ROWS == 1) {
      __syncthreads();
      if (tid < M) {
        float t = 0.f;
        for (int c = 0; c < band; ++c) t += sq[tid * band + c];
        rows.sums[tid * gridDim.x + blockIdx.x] = t;
      }
    }
  };
  for (int idx = tid; idx < band * M; idx += 512) {
    const int m = idx / band, lr = idx - m * band;
    const int n = b0 + lr, qd = lr >> 2, i = lr & 3;
    float a = 0.f, u = 0.f;
#pragma unroll
    for (int k = 0; k < SM_KW; ++k) {
      a += red[k][qd][i][m];
      if (sg_paired(EPI)) u += red[k][qg + qd][i][m];
    }
    if constexpr (NORM) {
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < SM_KW; ++k) s += ssw[k][m];
      const float inv = rsqrtf(s / (float)K + eps);
      a *= inv;
      u *= inv;
    }
    if constexpr (ROWS == 2) {
      const float inv = 1.0f / sqrtf(ssw[0][m] / (float)K + eps);
      a *= inv;
      u *= inv;
    }
    const bool first = idx == tid;
    if constexpr (FP8) {
      a *= first ? pre_sa : wscale[n];
      if (sg_paired(EPI)) u *= first ? pre_su : wscale[N + n];
    }
    if (G > 1) {   // device-coherent stores (write-through past the XCD's L2): read back by another workgroup
      const int wrows = (sg_paired(EPI)) ? 2 * N : N;
      float* slab = part + ((size_t)g * M + m) * wrows;
      __hip_atomic_store(slab + n, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (sg_paired(EPI)) __hip_atomic_store(slab + N + n, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      continue;
    }
    store(idx, m, n, a, u);
  }
  if (G == 1) row_sums();
  if (G == 1 || tickets == nullptr) return;   // (no tickets: sgemv_finalize_kernel sums the slabs)

  // ---- k-groups: the LAST workgroup of this band to finish sums the G slabs (fixed order, as the finalize kernel
  // would) and stores the result -- no second launch.  No cache-wide fences: the slab stores above are device-coherent
  // (write-through), every wave waits for its own stores to land before the workgroup counts its arrival with one
  // device-scope add, and the last workgroup reads the slabs with device-coherent loads.
  __shared__ int sm_last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's slab stores have landed
  __syncthreads();
  if (tid == 0)
    sm_last = __hip_atomic_fetch_add(&tickets[blockIdx.x], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
              (unsigned)(G - 1);
  __syncthreads();
  if (!sm_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");   // (compiler ordering: the loads stay below the add)
  const int wrows = (sg_paired(EPI)) ? 2 * N : N;
  for (int idx = tid; idx < band * M; idx += 512) {
    const int m = idx / band, n = b0 + idx - m * band;
    float a = 0.f, u = 0.f;
    for (int k = 0; k < G; ++k) {
      const float* slab = part + ((size_t)k * M + m) * wrows;
      a += __hip_atomic_load(slab + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (sg_paired(EPI)) u += __hip_atomic_load(slab + N + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    store(idx, m, n, a, u);
  }
  row_sums();
  if (tid == 0)   // ready for the next launch that draws this ticket range
    __hip_atomic_store(&tickets[blockIdx.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int EPI, bool RES>
__global__ void sgemv_finalize_kernel(void* __restrict__ out, const float* __restrict__ part, const bf16_t* res,
                                      int M, int N, int G, EpiAct act) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * N) return;
  const int m = i / N, n = i - m * N;
  const int wrows = sg_paired(EPI) ? 2 * N : N;
  float a = 0.f, u = 0.f;
  for (int g = 0; g < G; ++g) {
    const float* slab = part + ((size_t)g * M + m) * wrows;
    a += slab[n];
    if (sg_paired(EPI)) u += slab[N + n];
  }
  sm_store<EPI, RES>(out, i, a, u, RES ? bf2f(res[i]) : 0.f, act);
}

// MFMA plan (smfma_kernel): JT register steps per wave (1, 2, 4, 8; a step = 16 chunks of every row of a quad),
// jw live steps, G k-groups.  Needs whole steps (K % 128 bf16, K % 256 fp8); one k-group covers 8 waves x 8 steps
// (8192 k) -- fp8 4 steps (8192 k: an fp8 step holds twice the x of a bf16 one).  9 - 16 rows take more groups where bands of
// 16 output rows leave CUs idle, as long as a wave keeps two steps and the depth pays for the reduction (2.3 us): us, 16 rows,
// one group -> the rule's: 2048 x 8192 16.5 -> 12.7, x 6144 14.1 -> 10.9, 1024 x 8192 16.3 -> 10.0.  Up to 8 rows narrower
// bands do better (sm_launch).  The norm prologue needs all of K in one group.
struct SmPlan {
  int jt, jw, g;
};
static int sm_cus();
static bool sm_plan(int M, int N, int K, bool fp8, bool norm, SmPlan& p) {
  const int epc = fp8 ? 16 : 8;
  if (K % (16 * epc) != 0) return false;
  const int c16 = K / (16 * epc), jmax = fp8 ? 4 : 8;
  int g = (c16 + SM_KW * jmax - 1) / (SM_KW * jmax);
  if (M > 8 && !fp8 && !norm && c16 >= 48)
    while ((N + 15) / 16 * g * 2 <= sm_cus() && c16 >= 4 * SM_KW * g) g *= 2;
  const int jw = (c16 + SM_KW * g - 1) / (SM_KW * g);
  p = {jw <= 1 ? 1 : (jw <= 2 ? 2 : (jw <= 4 ? 4 : 8)), jw, g};
  return true;
}
// rows from which the matrix-core form takes over from the register dot2 form (K8S_SGEMV_MFMA_MIN_M, default 3:
// every sgemv row count -- at 4 rows it ties or beats the dot2 form, profiles/sgemv_mfma4_kernel_trace_r4.txt; 5
// keeps 3..4 rows on dot2; 17 turns it off: 9..16 rows then go back to mgemm).  The dot2 form remains the path
// for K that is not a whole number of 16-chunk steps.
static int sm_min_m() {
  static const int v = [] { const char* e = getenv("K8S_SGEMV_MFMA_MIN_M"); return e ? atoi(e) : 3; }();
  return v;
}
static int sm_cus() {
  static const int v = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                 hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  return v;
}
static bool sm_take(int M, int N, int K, bool fp8, bool norm, SmPlan& p) {
  return M >= sm_min_m() && M <= 16 && sm_plan(M, N, K, fp8, norm, p);
}

// Workgroups of the MFMA form per CU the band is sized for: what the kernel's registers allow (one for every form
// since the epilogue prefetch took the 8-row kernels past 128 VGPRs), capped by K8S_SGEMV_WG_PER_CU (default 1: at 2 the 70B QKV / gate/up / down ran 9 / 3 / 3 %
// slower -- twice the workgroups re-read x -- and O 3 % faster; profiles/sgemv_mfma4_kernel_trace_r4.txt).
static int sm_wg_cap() {
  static const int v = [] { const char* e = getenv("K8S_SGEMV_WG_PER_CU"); return e ? max(1, atoi(e)) : 1; }();
  return v;
}
static std::atomic<unsigned> g_sm_next_range{0};   // of this unit's ranges, for every instantiation (launches on any stream)

template <int MT, int JT, int EE, bool NN, bool RR, bool F8, int ROWS = 0>
static bool sm_launch(void* out, void* partial, const bf16_t* x, const void* W, const float* wscale, const bf16_t* res,
                      int M, int N, int K, float eps, const SmPlan& sp, hipStream_t stream, EpiAct act = {},
                      const SmRows& rows = {}, int* bands = nullptr) {
  static const int occ = [] {
    int n = 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(&smfma_kernel<MT, JT, EE, NN, RR, F8, ROWS>),
                                                     512, 0) != hipSuccess)
      n = 1;
    return max(1, min(n, sm_wg_cap()));
  }();
  // ~occ workgroups per CU and k-group, at least 8 rows (x is re-read per workgroup), at most the LDS partials'
  // quads (SwiGLU: gate + up quads, with the phantom rounding).  us with at least 16 rows -> 8 (8 x 2048 x 8192: in two k-groups
  // 11.2): 8 x 2048 x 8192 12.8 -> 9.5, x 4096 7.7 -> 6.1, x 2048 5.2 -> 4.8; 4 x 2048 x 8192 11.4 -> 8.8; 16 x 2048 x 4096 9.5 ->
  // 7.5, x 2048 6.4 -> 5.9
  constexpr int qmax = 512 / MT;
  const int bandmax = 4 * qmax / (sg_paired(EE) ? 2 : 1);
  const int per = max(1, sm_cus() * occ / sp.g);
  int band = max(min(8, N), (N + per - 1) / per);
  if (band > bandmax) {
    int nb = (N + bandmax - 1) / bandmax;
    nb = (nb + per - 1) / per * per;   // whole rounds of workgroups
    band = (N + nb - 1) / nb;
  }
  if constexpr (ROWS == 3) {   // bands of one input each, about a workgroup per CU
    band = 8;
    while (2 * band <= bandmax && rows.count % (2 * band) == 0 && (N + band - 1) / band > sm_cus() + sm_cus() / 8) band *= 2;
    if (rows.count % band != 0) return false;
  }
  const dim3 grid((N + band - 1) / band, sp.g);
  float* part = sp.g > 1 ? (float*)partial : nullptr;
  unsigned* tk = nullptr;   // k-groups: the in-kernel reduction's ticket range (rotating), if the bands fit one
  if (sp.g > 1 && grid.x <= (unsigned)SM_TICKET_RANGE) {
    unsigned* base = nullptr;
    if (hipGetSymbolAddress((void**)&base, HIP_SYMBOL(sm_tickets)) == hipSuccess)
      tk = base + (size_t)(g_sm_next_range.fetch_add(1) % SM_TICKET_RANGES) * SM_TICKET_RANGE;
  }
  if (bands != nullptr) *bands = (int)grid.x;
  if constexpr (ROWS != 0)   // (its sums have SM_SUMS places, the reduction by a second launch knows no rows)
    if ((ROWS == 1 && grid.x > (unsigned)SM_SUMS) || (sp.g > 1 && tk == nullptr)) return false;
  smfma_kernel<MT, JT, EE, NN, RR, F8, ROWS><<<grid, 512, 0, stream>>>(out, part, x, W, wscale, res, M, N, K, eps, band,
                                                                       sp.jw, tk, act, rows);
  return ROWS != 0 || tk != nullptr;
}

}  // namespace k8sllm
