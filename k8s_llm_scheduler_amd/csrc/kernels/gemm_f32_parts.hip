// fp32 products on the bf16 matrix cores: C[M, N] = A[M, K] W[N, K]^T, fp32 in and out, K % 32 == 0.
//
// A value of 24 bits is the sum of three bf16 of 8 (high, middle, low: each the rounding of what the ones before leave, so exact),
// and of the nine products of two such sums the six of 2^-16 and more are taken, the small ones first: what is left out is 2^-24 of
// a product and less, as much as one rounding of its fp32 sum.  Six bf16 products take 3 / 8 of the time of the fp32 one (2.5
// PFLOP/s over 157 TFLOP/s, over 6).  Registers sum chains of 64 k (128 from 128 steps on), and a second set the chains, so the
// error against 64 bits is below the fp32 pipes' (2-norm, here / there: K = 1024 1.2e-7 / 1.6 - 2.1e-7, 2048 1.2 - 1.5e-7 / 2.1 -
// 2.9e-7, 8192 1.5 - 1.6e-7 / 2.2 - 5.7e-7, 14336 1.7 - 2.25e-7 / 2.3 - 7.7e-7; one chain for all of K = 2048: 2.4 - 7e-7).
// Parts of infinities are NaN, a high part may round to infinity, and parts and products below 2^-126 may be lost: of a product at
// most 2^-126 times the other side's value, and six times 2^-126.  So an output is computed again with plain fp32 FMAs where it is not
// finite, where it is smaller than K 2^-97 times the largest value of its row and column (or 1: above that what may be lost is 2^-25
// of it and less), and where it is zero though both have values.  The largest values are met on the way to the parts, one
// instruction for two of them.  A wave computes such an output together: one does not show (a sum may happen to be zero, one in 10^7 or
// 10^8), 333 x 2048 x 8192 with a NaN in one row takes 161 us instead of 105, with an infinity in a column 145, and 1.8 ms where all
// outputs are zero.
//
// A workgroup of 8 waves owns 16 CW WC columns x 16 FQ rows: WC waves side by side, each with CW x 16 columns and all rows, and
// 8 / WC shares of k (steps of 32 k in turn).  A wave loads its weights itself and cuts them in registers; with WC > 1 the rows are
// cut once a workgroup and pass through LDS, with WC = 1 a wave cuts its own.  Both for the step after the current one, two
// values between every CW products (the barriers of the compiler's schedule keep them there: left alone it cuts everything first).
// Bound by the matrix cores on the large tiles (333 x 16384 x 2048, 142 us: 1.09 PFLOP/s of bf16 products with the padding, where
// large bf16 products reach 1.35), on the small ones by the loads of rows 64 bytes at a time and the cutting (60 x 2048 x 8192, 47 us: 27
// without the loads, 17 without both; loads two and four steps ahead, and tiles that start at different k, change nothing).
// us, fp32 pipes / here, weights from memory: 333 x 16384 x 2048 195 / 142, x 2048 x 8192 110 / 104, x 3072 x 2048 51 / 39, 512 x
// 16384 x 2048 257 / 168, 457 x 4096 x 14336 472 / 347, 150 x 28672 x 4096 338 / 253, 64 x 16384 x 2048 44 / 40, 17 x 2048 x 2048
// 14.8 / 11.1, 1 x 2048 x 8192 64 / 27, 16 x 3072 x 2048 18.6 / 11.1.  The largest values cost 1 - 3 % of that.
#include <math.h>

#include "common.h"

namespace k8sllm {

struct PartsArgs {
  float* C;
  const float *A, *W;
  int M, N, K, mt, nt, batch;
  long lda, ldw, ldc, sA, sW, sC;
  const int *a_rows, *tiles;        // listed tiles of at most 64 rows: 64 / Q blocks for each
  int vec;                          // 4 consecutive columns can be stored as one vector
  int chain;                        // steps of a chain - 1 (a power of two less one)
  float least;                      // of an output, over the larger side's largest value (or 1): below it parts may be missing
};

struct Three {                      // the parts of 8 values, two in a word
  u32x4 h, m, l;
};

// values 2 q and 2 q + 1 of the eight (a, b); top: the largest magnitude met so far
__device__ __forceinline__ void cut2(Three& t, const f32x4 (&r)[2], int q, float& top) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  float a = r[q >> 1][2 * q & 3], b = r[q >> 1][(2 * q & 3) + 1];
  asm volatile("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top), "+v"(a), "+v"(b));
  f32x2 x = {a, b};
  uint32_t p[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bf16x2 y = __builtin_convertvector(x, bf16x2);
    p[i] = __builtin_bit_cast(uint32_t, y);
    x = x - f32x2{lo_bf(p[i]), hi_bf(p[i])};
  }
  asm volatile("" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]));
  t.h[q] = p[0], t.m[q] = p[1], t.l[q] = p[2];
}
__device__ __forceinline__ Three cut(const f32x4 (&r)[2], float& top) {
  Three t;
#pragma unroll
  for (int q = 0; q < 4; ++q) cut2(t, r, q, top);
  return t;
}

template <int WC, int CW, int FQ>
__global__ __launch_bounds__(512, 2) void gemm_f32_parts_kernel(PartsArgs a) {
  constexpr int WK = 8 / WC, P = 16 * CW * WC, Q = 16 * FQ, NX = (FQ + WC - 1) / WC;
  constexpr int GS = Q * 16 + 32, BUF = WK * 12 * GS, RED = 8 * CW * FQ * 1024;
  constexpr int STAGES = WC > 1 ? 2 * BUF : 0, TOPS = WK * (P + Q) * 4 + 32, LDS = STAGES > RED + TOPS ? STAGES : RED + TOPS;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  const int tot = a.mt * a.nt * a.batch, q8 = tot >> 3, r8 = tot & 7, xcd = blockIdx.x & 7;
  int t = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (int)(blockIdx.x >> 3);
  const int ti = t % a.mt;
  t /= a.mt;
  const int tj = t % a.nt, tb = t / a.nt;
  const float *A = a.A + (size_t)tb * a.sA, *W = a.W + (size_t)tb * a.sW;
  int row0 = ti * Q, rows = min(Q, a.M - row0);
  if (a.tiles != nullptr) {
    constexpr int PER = 64 / Q > 0 ? 64 / Q : 1;
    const int y = ti / PER, sub = (ti - y * PER) * Q, grp = a.tiles[3 * y];
    if (grp < 0) return;
    row0 = a.tiles[3 * y + 1] + sub;
    rows = min(Q, a.tiles[3 * y + 2] - sub);
    if (rows <= 0) return;
    W += (size_t)grp * a.sW;
  }
  const auto row = [&](int r) { return A + (size_t)(a.a_rows != nullptr ? a.a_rows[row0 + r] : row0 + r) * a.lda; };
  const int col0 = tj * P;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, g = lane >> 4;
  const int wc = wid % WC, wk = wid / WC;
  const int S = a.K / 32, T = (S + WK - 1) / WK;
  const float* wp[CW];
#pragma unroll
  for (int c = 0; c < CW; ++c) wp[c] = W + (size_t)min(col0 + 16 * (wc * CW + c) + li, a.N - 1) * a.ldw + 4 * g;
  f32x4 wr[CW][2];
  auto load_w = [&](int s, int c) {
    const size_t k = 32 * (size_t)min(s * WK + wk, S - 1);
    wr[c][0] = *reinterpret_cast<const f32x4*>(wp[c] + k);
    wr[c][1] = *reinterpret_cast<const f32x4*>(wp[c] + k + 16);
  };
  // rows: with WC > 1 chunk tid + 512 n of the step's [k group][row][8 of 32], else this wave's own fragments
  constexpr int NR = WC > 1 ? NX : FQ;
  f32x4 xr[NR][2];
  const float* xp[NR];
  int xk[NR], xo[NR];
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    if constexpr (WC > 1) {
      const int c = min(tid + 512 * n, WK * Q * 4 - 1), q = c >> 2, r = q % Q;     // threads past the last chunk write it again, the same values
      xk[n] = q / Q;
      xp[n] = row(min(r, rows - 1)) + 4 * (c & 3);
      xo[n] = xk[n] * 12 * GS + (c & 3) * GS + r * 16;
    } else {
      xk[n] = wk, xo[n] = 0;
      xp[n] = row(min(16 * n + li, rows - 1)) + 4 * g;
    }
  }
  auto load_x = [&](int s, int n) {
    const size_t k = 32 * (size_t)min(s * WK + xk[n], S - 1);
    xr[n][0] = *reinterpret_cast<const f32x4*>(xp[n] + k);
    xr[n][1] = *reinterpret_cast<const f32x4*>(xp[n] + k + 16);
  };
  auto store_x = [&](int s, int n, const Three& p) {
    char* o = lds + (s & 1) * BUF + xo[n];
    *reinterpret_cast<u32x4*>(o) = p.h;
    *reinterpret_cast<u32x4*>(o + 4 * GS) = p.m;
    *reinterpret_cast<u32x4*>(o + 8 * GS) = p.l;
  };
  auto meet = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  f32x4 acc[CW][FQ], sum[CW][FQ];
#pragma unroll
  for (int c = 0; c < CW; ++c)
#pragma unroll
    for (int j = 0; j < FQ; ++j) acc[c][j] = sum[c][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  Three wa[CW], wb[CW], xf[2], xs;
  float wtop[CW], xtop[NR];         // the largest magnitudes of this lane's share of a column, of a row
#pragma unroll
  for (int c = 0; c < CW; ++c) wtop[c] = 0.f;
#pragma unroll
  for (int n = 0; n < NR; ++n) xtop[n] = 0.f;
  const auto read_x = [&](int s, int j) {
    const char* xb = lds + (s & 1) * BUF + wk * 12 * GS + g * GS + li * 16 + j * 256;
    return Three{*reinterpret_cast<const u32x4*>(xb), *reinterpret_cast<const u32x4*>(xb + 4 * GS),
                 *reinterpret_cast<const u32x4*>(xb + 8 * GS)};
  };
#pragma unroll
  for (int c = 0; c < CW; ++c) load_w(0, c);
#pragma unroll
  for (int n = 0; n < NR; ++n) load_x(0, n);
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    wa[c] = cut(wr[c], wtop[c]);
    load_w(1, c);
  }
  if constexpr (WC > 1) {
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      store_x(0, n, cut(xr[n], xtop[n]));
      load_x(1, n);
    }
    meet();
  } else {
    xf[0] = cut(xr[0], xtop[0]);
    load_x(1, 0);
  }
  // One step's products.  `more`: between them the next step's weights and rows are cut into parts, two values at a time, and the
  // loads behind them go out.
  const auto step = [&](auto more, int s, const Three* w, Three* wn) {
    constexpr bool MORE = decltype(more)::value;
    constexpr int GROUPS = 6 * FQ, WP = 4 * CW, XP = 4 * NX;
    if constexpr (WC > 1) xf[0] = read_x(s, 0);
#pragma unroll
    for (int j = 0; j < FQ; ++j) {
      Three& x = xf[(WC > 1 || FQ % 2 == 0) ? j & 1 : 0];
      Three& xn = xf[(WC > 1 || FQ % 2 == 0) ? (j & 1) ^ 1 : 1];
      if (WC > 1 && j + 1 < FQ) xn = read_x(s, j + 1);
#pragma unroll
      for (int p = 0; p < 6; ++p) {
#pragma unroll
        for (int c = 0; c < CW; ++c)
          acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, p == 0 ? w[c].l : p == 2 || p == 3 ? w[c].m : w[c].h),
              __builtin_bit_cast(bf16x8, p == 1 ? x.l : p == 2 || p == 4 ? x.m : x.h), acc[c][j], 0, 0, 0);
#pragma unroll
        for (int c = 0; c < CW; ++c) asm volatile("" : "+v"(acc[c][j]));
        const int q = 6 * j + p;
        if constexpr (MORE) {
#pragma unroll
          for (int n = 0; n < WP; ++n)
            if (n * GROUPS / WP == q) {
              cut2(wn[n >> 2], wr[n >> 2], n & 3, wtop[n >> 2]);
              if ((n & 3) == 3) load_w(s + 2, n >> 2);
            }
        }
        if constexpr (WC > 1 && MORE) {
#pragma unroll
          for (int n = 0; n < XP; ++n)
            if (n * GROUPS / XP == q) {
              cut2(xs, xr[n >> 2], n & 3, xtop[n >> 2]);
              if ((n & 3) == 3) {
                store_x(s + 1, n >> 2, xs);
                load_x(s + 2, n >> 2);
              }
            }
        }
        if constexpr (WC == 1) {
          const int n = j + 1 < FQ ? j + 1 : 0;
          if (p < 4 && (MORE || n)) {
            cut2(xn, xr[n], p, xtop[n]);
            if (p == 3 && MORE) load_x(n ? s + 1 : s + 2, n);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (WC == 1 && FQ % 2 == 1) xf[0] = xf[1];
    }
  };
  const auto flush = [&]() {
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        sum[c][j] += acc[c][j];
        acc[c][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  const auto go = [&](int s, const Three* w, Three* wn) {
    step(std::true_type{}, s, w, wn);
    if ((s & a.chain) == a.chain) flush();
    if constexpr (WC > 1) meet();
  };
  const bool last = (T - 1) * WK + wk < S;        // the last step's share of k may be empty
  int s = 0;
  for (; s + 2 < T; s += 2) {
    go(s, wa, wb);
    go(s + 1, wb, wa);
  }
  if (s + 2 == T) {
    go(s, wa, wb);
    if (last) step(std::false_type{}, s + 1, wb, wa);
  } else if (last) {
    step(std::false_type{}, s, wa, wb);
  }
  flush();
  float* C = a.C + (size_t)tb * a.sC;
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int c = 0; c < CW; ++c)
#pragma unroll
    for (int j = 0; j < FQ; ++j) *reinterpret_cast<f32x4*>(red + (((wid * CW + c) * FQ + j) * 64 + lane) * 4) = sum[c][j];
  // [wave]: its largest of all; [share of k][column], [row]
  float *tops = red + RED / 4, *wtops = tops + 8, *xtops = wtops + WK * P;
  float most = 0.f;
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    const float m = lane_max<16>(lane_max<32>(wtop[c]));
    most = fmaxf(most, wtop[c]);
    if (g == 0) wtops[wk * P + 16 * (wc * CW + c) + li] = m;
  }
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    most = fmaxf(most, xtop[n]);
    if constexpr (WC > 1) {
      const float m = lane_max<1>(lane_max<2>(xtop[n]));      // a row's four chunks
      const int q = (tid + 512 * n) >> 2;                     // (its rows in turn: a share of k has Q of them)
      if ((tid & 3) == 0 && q < WK * Q) xtops[q] = m;
    } else {
      const float m = lane_max<16>(lane_max<32>(xtop[n]));
      if (g == 0) xtops[wk * Q + 16 * n + li] = m;
    }
  }
  most = wave_max(most);
  if (lane == 0) tops[wid] = most;
  __syncthreads();
  // most outputs are large enough for any value of the workgroup
  const f32x4 t0 = *reinterpret_cast<const f32x4*>(tops), t1 = *reinterpret_cast<const f32x4*>(tops + 4);
  most = fmaxf(fmaxf(fmaxf(t0[0], t0[1]), fmaxf(t0[2], t0[3])), fmaxf(fmaxf(t1[0], t1[1]), fmaxf(t1[2], t1[3])));
  const float enough = a.least * fmaxf(most, 1.f);
#pragma unroll 1
  for (int f = wk; f < CW * FQ; f += WK) {
    f32x4 y = *reinterpret_cast<const f32x4*>(red + ((wc * CW * FQ + f) * 64 + lane) * 4);
#pragma unroll
    for (int k = 1; k < WK; ++k) y += *reinterpret_cast<const f32x4*>(red + (((k * WC + wc) * CW * FQ + f) * 64 + lane) * 4);
    const int r = 16 * (f % FQ) + li, n = col0 + 16 * (wc * CW + f / FQ) + 4 * g;
    const bool mine = r < rows && n < a.N;
    uint32_t again = 0;             // bit e: this lane's output n + e
#pragma unroll
    for (int e = 0; e < 4; ++e) again |= (mine && n + e < a.N && !(fabsf(y[e]) >= enough && fabsf(y[e]) < INFINITY)) << e;
    if (__any(again != 0)) {
      if (again != 0) {
        float mx = 0.f;
        f32x4 mw = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < WK; ++k) {
          mx = fmaxf(mx, xtops[k * Q + r]);
#pragma unroll
          for (int e = 0; e < 4; ++e) mw[e] = fmaxf(mw[e], wtops[k * P + n - col0 + e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (y[e] == 0.f ? !(mx > 0.f && mw[e] > 0.f) : fabsf(y[e]) >= a.least * fmaxf(fmaxf(mx, mw[e]), 1.f) && fabsf(y[e]) < INFINITY)
            again &= ~(1u << e);
      }
      // the wave takes one output after the other, 256 of k at a time
#pragma unroll 1
      for (int e = 0; e < 4; ++e)
#pragma unroll 1
        for (uint64_t left = __ballot(again >> e & 1); left != 0; left &= left - 1) {
          const int src = __builtin_ctzll(left);
          const float* x = row(16 * (f % FQ) + (src & 15));
          const float* w = W + (size_t)(col0 + 16 * (wc * CW + f / FQ) + 4 * (src >> 4) + e) * a.ldw;
          float v = 0.f;
#pragma unroll 4
          for (int k = 4 * lane; k < a.K; k += 256) {
            const f32x4 xk = *reinterpret_cast<const f32x4*>(x + k), wv = *reinterpret_cast<const f32x4*>(w + k);
#pragma unroll
            for (int i = 0; i < 4; ++i) v = fmaf(xk[i], wv[i], v);
          }
          v = wave_sum(v);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (lane == src && i == e) y[i] = v;
        }
    }
    if (!mine) continue;
    const size_t at = (size_t)(row0 + r) * a.ldc + n;
    if (a.vec) {
      *reinterpret_cast<f32x4*>(C + at) = y;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < a.N) C[at + e] = y[e];
    }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" double k8s_gemm_f32_cost(int M, int N, int K, int batch);

// The tile (100 WC + 10 CW + FQ) for a product, 0: the fp32 pipes' kernels are expected to be as fast.  A tile's time is 4 us, a round's
// steps and start for every round of workgroups over the CUs (from three on two of the small ones share one), and a share of what the weights
// take; fitted to M 1 - 512, N 128 - 32768, K 512 - 14336 (rms error 4 - 7 % of the larger ones, 10 - 17 % of those of one column of waves), as are the fp32
// pipes' times.  A tenth is left to these: of 300 sizes none is slower by more than 3 %, and all take 23 % less on average, 0.8 % more than
// with the best of both for each (with the largest values met, of 169 more that it takes one by 2 %, 31 % less on average).  They keep 33 - 100 rows of 1024 - 4096 columns in one round (56 x 3072 x 2048 16.1 / 19.3, 40 x 4096 x 14336 88 / 108), short weights (24 x 1024 x 512 6.5 / 7.3) and
// few rows of wide ones, which both read at the memory's rate (3 x 32768 x 2048 40 / 42).
// Listed tiles: from 32 rows a group on, where the groups' tiles of 32 or 64 rows of 64 columns fill one round, else 64 x 128.  Groups x columns x k, rows
// a group: 8 x 4096 x 2048, 40 90 / 66, 250 287 / 226; 8 x 2048 x 2048, 40 58 / 37; 16 x 1024 x 2048, 40 45 / 38; 4 x 2048 x 2048, 40 32
// / 25; 9 x 4096 x 2048, 40 109 / 102, 24 84 / 96; 8 x 4096 x 2048, 16 61 / 66.
extern "C" int k8s_gemm_f32_parts_rule(int M, int N, int K, int batch, int ntiles) {
  if (K < 512 || K % 32 || M <= 0 || N <= 0 || batch <= 0) return 0;
  if (ntiles > 0) {
    const long groups = ntiles - (M + 63) / 64 > 1 ? ntiles - (M + 63) / 64 : 1;
    if (M < 32 * groups || K < 1024 || N < 512) return 0;
    const double t = (M <= 48 * groups ? groups : M / 64.0 + groups / 2.0) * ((N + 63) / 64);
    return t <= 128.0 && M <= 48 * groups ? 222 : t <= 256.0 ? 224 : 424;
  }
  static const struct { int tile; float step, start, weights; } menu[] = {
      {111, 0.87f, 0.5f, 0.f},    {112, 1.06f, 2.0f, 0.f},    {121, 1.27f, 0.7f, 0.006f}, {122, 1.63f, 1.1f, 0.f},    {222, 1.02f, 0.8f, 0.039f},
      {223, 1.34f, 0.9f, 0.042f}, {224, 1.55f, 1.1f, 0.046f}, {225, 1.81f, 1.6f, 0.054f}, {226, 2.00f, 1.6f, 0.057f}, {423, 1.11f, 0.7f, 0.045f},
      {424, 1.24f, 0.8f, 0.051f}, {425, 1.62f, 1.4f, 0.052f}, {426, 1.69f, 2.0f, 0.056f}, {427, 1.86f, 2.1f, 0.060f}, {826, 1.51f, 2.4f, 0.061f},
      {827, 1.70f, 3.1f, 0.055f}, {828, 1.86f, 3.4f, 0.054f}};
  double best = 0.9 * k8s_gemm_f32_cost(M, N, K, batch);
  int pick = 0;
  for (const auto& m : menu) {
    const int wc = m.tile / 100, p = 16 * (m.tile / 10 % 10) * wc, q = 16 * (m.tile % 10);
    const double n = (double)((M + q - 1) / q) * ((N + p - 1) / p) * batch / 256.0;
    const double t = 4.0 + (m.tile < 122 && n > 2.0 ? n : ceil(n)) * (m.step * ((K / 32 * wc + 7) / 8) + m.start) +
                     m.weights * 4e-6 * N * (double)K * batch;
    if (t < best) {
      best = t;
      pick = m.tile;
    }
  }
  return pick;
}

// tile: one of the menu's; listed tiles of at most 64 rows: with FQ 1, 2 or 4.
extern "C" int k8s_gemm_f32_parts(float* C, const float* A, const float* W, int M, int N, int K, long lda, long ldw, long ldc,
                                  int batch, long sA, long sW, long sC, const int* a_rows, const int* tiles, int ntiles,
                                  int tile, hipStream_t s) {
  const int wc = tile / 100, cw = tile / 10 % 10, fq = tile % 10;
  if (M <= 0 || N <= 0 || K < 32 || K % 32 || batch <= 0 || wc < 1 || cw < 1 || fq < 1 || (lda | ldw | sA | sW) % 4 ||
      (((uintptr_t)A | (uintptr_t)W) & 15))
    return -1;
  if (tiles != nullptr && (64 % (16 * fq) || ntiles <= 0)) return -1;
  PartsArgs a = {C, A, W, M, N, K, 0, 0, 0, lda, ldw, ldc, sA, sW, sC, a_rows, tiles, 0, 0, (float)K * 0x1p-97f};
  a.mt = tiles != nullptr ? ntiles * (4 / fq) : (M + 16 * fq - 1) / (16 * fq);
  a.nt = (N + 16 * cw * wc - 1) / (16 * cw * wc);
  a.batch = tiles != nullptr ? 1 : batch;
  const long long blocks = (long long)a.mt * a.nt * a.batch;
  if (blocks > (1LL << 30)) return -2;
  a.vec = N % 4 == 0 && ldc % 4 == 0 && sC % 4 == 0 && ((uintptr_t)C & 15) == 0;
  // chains of 2 steps, of 4 where they would be more than 64 (457 x 4096 x 14336, 64 x 128 tiles, 224 steps: 2.36e-7, 2.25e-7)
  a.chain = (long)K * wc > 32 * 8 * 128 ? 3 : 1;
#define K8S_FP(WC, CW, FQ)                                                                \
  case 100 * WC + 10 * CW + FQ:                                                           \
    gemm_f32_parts_kernel<WC, CW, FQ><<<dim3((unsigned)blocks), 512, 0, s>>>(a);          \
    break;
  switch (tile) {
    K8S_FP(1, 1, 1)
    K8S_FP(1, 1, 2)
    K8S_FP(1, 2, 1)
    K8S_FP(1, 2, 2)
    K8S_FP(2, 2, 2)
    K8S_FP(2, 2, 3)
    K8S_FP(2, 2, 4)
    K8S_FP(2, 2, 5)
    K8S_FP(2, 2, 6)
    K8S_FP(4, 2, 3)
    K8S_FP(4, 2, 4)
    K8S_FP(4, 2, 5)
    K8S_FP(4, 2, 6)
    K8S_FP(4, 2, 7)
    K8S_FP(8, 2, 6)
    K8S_FP(8, 2, 7)
    K8S_FP(8, 2, 8)
    default: return -1;
  }
#undef K8S_FP
  return (int)hipGetLastError();
}
