// fp32 residual stream: embedding rows, fused residual-add + RMS norm, gated activations, and a GEMM for any shape.
//
// Models whose residual sum lives in fp32 keep x as [T, W] floats; every branch output (bf16, or fp32 in the all-fp32
// mode) is added in fp32 by the norm that follows it, so the add costs no extra pass.  All kernels take the
// activation / weight element type as a template parameter: bf16 storage or true fp32.
#include "common.h"
#include "latent_row.h"

namespace k8sllm {

// out[t, :] = float(table[ids[t], :]) * scale; copy (optional) the same in the table's type, as the first sublayer reads it
template <typename TA>
__device__ __forceinline__ void embed_row(float* __restrict__ out, TA* __restrict__ copy, const int* __restrict__ ids,
                                          const TA* __restrict__ table, int W, int vocab, float scale, int t) {
  int id = ids[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const float v = ldf(table, (size_t)id * W + i) * scale;
    out[(size_t)t * W + i] = v;
    if (copy != nullptr) stf(copy, (size_t)t * W + i, v);
  }
}
template <typename TA>
__global__ void embed_rows_kernel(float* __restrict__ out, TA* __restrict__ copy, const int* __restrict__ ids,
                                  const TA* __restrict__ table, int W, int vocab, float scale) {
  embed_row(out, copy, ids, table, W, vocab, scale, blockIdx.x);
}

// What a step of single tokens needs to know of its B slot rows, in one launch: pos = ctx - 1, the cache slot of that
// position (-1: an idle row, ctx <= 0), ar = 0 .. B (query offsets, sequence and state slot of every row).  A context
// beyond its row of the block table idles the row.  Launch bound: as a dozen element-wise launches this took 67 us of a
// captured step (4.6 us a launch), as one 5 us.
__device__ __forceinline__ void decode_meta_row(int* __restrict__ pos, int* __restrict__ slots, int* __restrict__ ar,
                                                const int* __restrict__ ctx, const int* __restrict__ block_tables, int max_blocks,
                                                int B, int bs, int i) {
  if (i > B) return;
  ar[i] = i;
  if (i == B) return;
  const int p = ctx[i] - 1, blk = p >= 0 ? p / bs : 0;
  const bool live = p >= 0 && blk < max_blocks;
  pos[i] = live ? p : min(p, -1);
  slots[i] = live ? block_tables[(size_t)i * max_blocks + blk] * bs + (p - blk * bs) : -1;
}
__global__ void decode_meta_kernel(int* __restrict__ pos, int* __restrict__ slots, int* __restrict__ ar,
                                   const int* __restrict__ ctx, const int* __restrict__ block_tables, int max_blocks,
                                   int B, int bs) {
  decode_meta_row(pos, slots, ar, ctx, block_tables, max_blocks, B, bs, blockIdx.x * blockDim.x + threadIdx.x);
}
// Both of a step of B tokens, which begin it, in one launch: workgroups of a row each, then those of the step's description.
template <typename TA>
__global__ void embed_step_kernel(float* __restrict__ out, TA* __restrict__ copy, const int* __restrict__ ids,
                                  const TA* __restrict__ table, int W, int vocab, float scale, int* __restrict__ pos,
                                  int* __restrict__ slots, int* __restrict__ ar, const int* __restrict__ ctx,
                                  const int* __restrict__ block_tables, int max_blocks, int B, int bs) {
  const int t = blockIdx.x;
  if (t < B) embed_row(out, copy, ids, table, W, vocab, scale, t);
  else decode_meta_row(pos, slots, ar, ctx, block_tables, max_blocks, B, bs, (t - B) * blockDim.x + threadIdx.x);
}

// x[t] += mult * (branch[t] + branch2[t]) + rowvec (each optional), stored back in fp32; then (w != null)
// out[t] = x[t] / sqrt(mean(x[t]^2) + eps) * (offset + w), the mean taken over each of `groups` equal consecutive parts
// of the row by itself.  One workgroup per row; groups > 1: one wave per part.
template <typename TA>
__global__ __launch_bounds__(256) void resnorm_kernel(float* __restrict__ x, const TA* __restrict__ branch,
                                                      const TA* __restrict__ branch2, float mult,
                                                      const TA* __restrict__ rowvec, const TA* __restrict__ w,
                                                      float offset, float eps, TA* __restrict__ out, int W, int groups) {
  __shared__ float red[16];
  const size_t base = (size_t)blockIdx.x * W;
  float ss = 0.f;
  const bool upd = branch != nullptr || rowvec != nullptr;
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    float v = x[base + i];
    if (branch != nullptr) v += mult * (ldf(branch, base + i) + (branch2 != nullptr ? ldf(branch2, base + i) : 0.f));
    if (rowvec != nullptr) v += ldf(rowvec, i);
    if (upd) x[base + i] = v;
    ss += v * v;
  }
  if (w == nullptr) return;
  if (groups <= 1) {
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)W + eps);
    for (int i = threadIdx.x; i < W; i += blockDim.x)
      stf(out, base + i, x[base + i] * inv * (offset + ldf(w, i)));
    return;
  }
  __syncthreads();   // the updated row is read back by other threads
  const int Wg = W / groups, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int g = wave; g < groups; g += nw) {
    const size_t b = base + (size_t)g * Wg;
    float sg = 0.f;
    for (int i = lane; i < Wg; i += 64) {
      const float v = x[b + i];
      sg += v * v;
    }
    sg = wave_sum(sg);
    const float inv = 1.0f / sqrtf(sg / (float)Wg + eps);
    for (int i = lane; i < Wg; i += 64) stf(out, b + i, x[b + i] * inv * (offset + ldf(w, (size_t)g * Wg + i)));
  }
}

// The form without groups for rows of whole vectors (W % 4 == 0, W <= 1024 NV, aligned pointers), w given: all loads ahead of
// the reduction, the row in registers.  Bound by memory for prompts and by latency for single rows: 2048 rows of 2048, bf16
// branch, 15.4 -> 10.4 us (50 MB: 6.3 us at 8 TB/s); 8 rows 7.7 -> 4.6 us.
template <typename TA, int NV>
__global__ __launch_bounds__(256) void resnorm_row_kernel(float* __restrict__ x, const TA* __restrict__ branch,
                                                          const TA* __restrict__ branch2, float mult,
                                                          const TA* __restrict__ rowvec, const TA* __restrict__ w,
                                                          float offset, float eps, TA* __restrict__ out, int W) {
  __shared__ float red[16];
  const size_t base = (size_t)blockIdx.x * W;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 xv[NV], bv[NV], cv[NV], rv[NV], wv[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int i = 4 * (threadIdx.x + 256 * n);
    const bool in = i < W;
    xv[n] = in ? ldf4(x + base + i) : zero;
    bv[n] = in && branch != nullptr ? ldf4(branch + base + i) : zero;
    cv[n] = in && branch2 != nullptr ? ldf4(branch2 + base + i) : zero;
    rv[n] = in && rowvec != nullptr ? ldf4(rowvec + i) : zero;
    wv[n] = in ? ldf4(w + i) : zero;
  }
  float ss = 0.f;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int i = 4 * (threadIdx.x + 256 * n);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = xv[n][e];
      if (branch != nullptr) v += mult * (bv[n][e] + cv[n][e]);
      if (rowvec != nullptr) v += rv[n][e];
      xv[n][e] = v;
      ss += v * v;
    }
    if (i < W && (branch != nullptr || rowvec != nullptr)) stf4(x + base + i, xv[n]);
  }
  ss = row_total(ss, red + 8);
  const float inv = 1.0f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int i = 4 * (threadIdx.x + 256 * n);
    if (i >= W) continue;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = xv[n][e] * inv * (offset + wv[n][e]);
    stf4(out + base + i, y);
  }
}

// A step of single tokens: the row's norm (resnorm_row_kernel) and the token shift that reads it in one launch, which a chain of small
// launches pays for twice: h = the norm's row, out[k] = h + (prev - h) mu[k] with prev the slot's row of `state` (zeros at position 0),
// which becomes h; an idle row (position < 0) gives zeros and leaves the state alone.  As resnorm_row_kernel and token_shift_row_kernel
// in turn, bit for bit.  A chain of latencies: 8 rows of 2048, five mixes, 4.1 + 4.5 us in two launches, 7.3 in one, and the gap between
// them.
constexpr int SHIFT_MIXES = 5;
template <typename TA, int NV>
__global__ __launch_bounds__(256) void norm_shift_kernel(TA* __restrict__ out, float* __restrict__ x, const TA* __restrict__ branch,
                                                         float mult, const TA* __restrict__ rowvec, const TA* __restrict__ w,
                                                         float offset, float eps, const TA* __restrict__ mu, TA* __restrict__ state,
                                                         const int* __restrict__ seq_slots, const int* __restrict__ positions, int n,
                                                         int T, int W) {
  __shared__ float red[4];
  const int t = blockIdx.x;
  const size_t base = (size_t)t * W;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  const int p = positions[t], slot = seq_slots[t];
  TA* row = state + (size_t)(p >= 0 ? slot : 0) * W;
  f32x4 xv[NV], bv[NV], rv[NV], wv[NV], pv[NV], mv[SHIFT_MIXES][NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int i = 4 * (threadIdx.x + 256 * q);
    const bool in = i < W;
    xv[q] = in ? ldf4(x + base + i) : zero;
    bv[q] = in && branch != nullptr ? ldf4(branch + base + i) : zero;
    rv[q] = in && rowvec != nullptr ? ldf4(rowvec + i) : zero;
    wv[q] = in ? ldf4(w + i) : zero;
#pragma unroll
    for (int k = 0; k < SHIFT_MIXES; ++k) mv[k][q] = in && k < n ? ldf4(mu + (size_t)k * W + i) : zero;
    pv[q] = in ? ldf4(row + i) : zero;             // (of a new sequence or an idle row: not used)
  }
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int i = 4 * (threadIdx.x + 256 * q);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = xv[q][e];
      if (branch != nullptr) v += mult * bv[q][e];
      if (rowvec != nullptr) v += rv[q][e];
      xv[q][e] = v;
      ss += v * v;
    }
    if (i < W && (branch != nullptr || rowvec != nullptr)) stf4(x + base + i, xv[q]);
  }
  ss = row_total(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int i = 4 * (threadIdx.x + 256 * q);
    if (i >= W) continue;
    f32x4 h, d;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = xv[q][e] * inv * (offset + wv[q][e]);
      if constexpr (sizeof(TA) == 2) h[e] = bf2f(f2bf(h[e]));
      d[e] = (p > 0 ? pv[q][e] : 0.f) - h[e];
    }
#pragma unroll
    for (int k = 0; k < SHIFT_MIXES; ++k) {
      if (k >= n) break;
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = p < 0 ? 0.f : h[e] + d[e] * mv[k][q][e];
      stf4(out + ((size_t)k * T + t) * W + i, y);
    }
    if (p >= 0) stf4(row + i, h);
  }
}

// Norm after the sum: x[t] <- (alpha x[t] + c1 branch[t] + c2 branch2[t]) / sqrt(mean(.^2) + eps) * gain, stored back
// in fp32 (the stream stays normed); `out` (optional) receives the same row in the activation type, for the sublayer
// that reads it next.  `gain` is one number for the whole row.  One workgroup per row; the row is held in registers
// (W <= 256 * 16) or re-formed from its inputs on the second pass.
template <typename TA>
__global__ __launch_bounds__(256) void postnorm_kernel(float* __restrict__ x, const TA* __restrict__ branch,
                                                       const TA* __restrict__ branch2, float alpha, float c1, float c2,
                                                       float gain, float eps, TA* __restrict__ out, int W) {
  __shared__ float red[16];
  const size_t base = (size_t)blockIdx.x * W;
  auto value = [&](int i) -> float {
    float v = alpha * x[base + i];
    if (branch != nullptr) v = fmaf(c1, ldf(branch, base + i), v);
    if (branch2 != nullptr) v = fmaf(c2, ldf(branch2, base + i), v);
    return v;
  };
  float ss = 0.f;
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const float v = value(i);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float m = gain / sqrtf(ss / (float)W + eps);
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const float y = value(i) * m;      // element i is read and written by this thread only
    x[base + i] = y;
    if (out != nullptr) stf(out, base + i, y);
  }
}

// Norm of a sublayer's output ahead of the sum: x[t] += branch[t] / sqrt(mean(branch[t]^2) + eps) * w, in fp32, the
// branch taken with its `bias` added (optional); `out` (optional) receives the new row in the activation type, for the
// sublayer that reads the stream next -- or (nw != null) its norm, x[t] / sqrt(mean(x[t]^2) + eps) * nw * gain, for a
// sublayer that is normed on both sides.  `dot` (optional, with nw): dot[t] = sum of the normed row times dotw, fp32 (a
// projection onto one number per token).  branch == null: nothing is added.  One workgroup per row.  NV > 0 (W % 4 == 0,
// W <= 1024 NV): everything a thread needs is loaded as vectors ahead of the reductions and stays in registers; else the
// row is read again after them (a thread re-reads only the elements it wrote).
// MOE (NV > 0): the branch is the experts' combine of moe.hip, branch[t] = sum over `top` choices k of scale D[pos[t, k]] + gate_t s_t,
// rounded to its type as that kernel's output is; s_t is row t of `shared` or, where that is null and pos has one column more, D's row
// pos[t, top] (shared and pos of `top` columns null: no shared expert), gate_t = sigmoid(logits[t ld]) (logits null: 1).  It saves
// the combine's launch and its output's way through memory: 32 rows of 2048 5.0 + 5.6 us in a step, 1534 rows 8.0 + 10.5.
template <typename TA>
struct MoeBranch {
  const TA* D;
  const int* pos;
  const TA* shared;
  const float* logits;
  int cols, top, ld;
  float scale;
};
template <typename TB, typename TA, int NV, bool MOE = false>
__global__ __launch_bounds__(256) void branchnorm_kernel(float* __restrict__ x, const TB* __restrict__ branch,
                                                         const TA* __restrict__ w, const TA* __restrict__ bias,
                                                         const TA* __restrict__ nw, float gain,
                                                         const TA* __restrict__ dotw, float* __restrict__ dot, float eps,
                                                         TA* __restrict__ out, int W, MoeBranch<TA> moe) {
  __shared__ float red[16];
  const size_t base = (size_t)blockIdx.x * W;
  float ss = 0.f, ds = 0.f;
  static_assert(!MOE || NV > 0, "the combine goes with whole vectors");
  const bool add = MOE || branch != nullptr;
  if constexpr (NV > 0) {
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 v[NV], xv[NV], wv[NV], nv[NV];
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int i = 4 * (threadIdx.x + 256 * n);
      const bool in = i < W;
      if constexpr (!MOE) v[n] = in && branch != nullptr ? ldf4(branch + base + i) : zero;
      xv[n] = in ? ldf4(x + base + i) : zero;
      wv[n] = in && add ? ldf4(w + i) : zero;
      nv[n] = in && nw != nullptr ? ldf4(nw + i) : zero;
    }
    if constexpr (MOE) {
      const int* pos = moe.pos + (size_t)blockIdx.x * moe.cols;
      const float gate = moe.logits != nullptr ? 1.f / (1.f + expf(-moe.logits[(size_t)blockIdx.x * moe.ld])) : 1.f;
      const TA* last = moe.shared != nullptr ? moe.shared + base : moe.cols > moe.top ? moe.D + (size_t)pos[moe.top] * W : nullptr;
#pragma unroll
      for (int n = 0; n < NV; ++n) v[n] = zero;
      for (int k = 0; k < moe.top; ++k) {
        const TA* row = moe.D + (size_t)pos[k] * W;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const int i = 4 * (threadIdx.x + 256 * n);
          const f32x4 d = i < W ? ldf4(row + i) : zero;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[n][e] = fmaf(moe.scale, d[e], v[n][e]);
        }
      }
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const int i = 4 * (threadIdx.x + 256 * n);
        if (last != nullptr) {
          const f32x4 d = i < W ? ldf4(last + i) : zero;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[n][e] = fmaf(gate, d[e], v[n][e]);
        }
        if constexpr (sizeof(TA) == 2) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[n][e] = bf_round(v[n][e]);
        }
      }
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int i = 4 * (threadIdx.x + 256 * n);
      if (i < W && bias != nullptr) {
        const f32x4 bv = ldf4(bias + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[n][e] += bv[e];
      }
    }
    if (add) {
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += v[n][e] * v[n][e];
      ss = row_total(ss, red + 8);
      const float inv = 1.0f / sqrtf(ss / (float)W + eps);
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const int i = 4 * (threadIdx.x + 256 * n);
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[n][e] = fmaf(v[n][e] * inv, wv[n][e], xv[n][e]);
        if (i < W) stf4(x + base + i, xv[n]);
      }
    }
    if (out == nullptr) return;
    float m = 1.f;
    if (nw != nullptr) {           // uniform
      ss = 0.f;
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += xv[n][e] * xv[n][e];
      ss = row_total(ss, red + 12);
      m = gain / sqrtf(ss / (float)W + eps);
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int i = 4 * (threadIdx.x + 256 * n);
      if (i >= W) continue;
      f32x4 y = xv[n];
      if (nw != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] *= m * nv[n][e];
      }
      stf4(out + base + i, y);
      if (dot != nullptr) {
        const f32x4 dv = ldf4(dotw + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) ds = fmaf(y[e], dv[e], ds);
      }
    }
  } else {
    auto value = [&](int i) -> float { return ldf(branch, base + i) + (bias != nullptr ? ldf(bias, i) : 0.f); };
    float inv = 0.f, s2 = 0.f;
    if (branch != nullptr) {
      for (int i = threadIdx.x; i < W; i += blockDim.x) {
        const float v = value(i);
        ss += v * v;
      }
      ss = block_sum(ss, red);
      inv = 1.0f / sqrtf(ss / (float)W + eps);
    }
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
      float y = x[base + i];
      if (branch != nullptr) {
        y = fmaf(value(i) * inv, ldf(w, i), y);
        x[base + i] = y;
      }
      s2 += y * y;
      if (out != nullptr && nw == nullptr) stf(out, base + i, y);
    }
    if (out == nullptr || nw == nullptr) return;
    s2 = block_sum(s2, red);
    const float m = gain / sqrtf(s2 / (float)W + eps);
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
      const float y = x[base + i] * m * ldf(nw, i);
      stf(out, base + i, y);
      if (dot != nullptr) ds = fmaf(y, ldf(dotw, i), ds);
    }
  }
  if (dot != nullptr) {            // uniform
    ds = block_sum(ds, red);
    if (threadIdx.x == 0) dot[blockIdx.x] = ds;
  }
}

// out[t, c] = y[t, c] * f(gate[t, c]) with f = sigmoid (kind 0) or silu (kind 1); y and gate are row-strided views.
template <typename TY, typename TA>
__global__ void gate_mul_kernel(TA* __restrict__ out, const TY* __restrict__ y, long ldy, const TA* __restrict__ gate,
                                long ldg, int T, int F, int kind) {
  const size_t n = (size_t)T * F;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const size_t t = i / F, c = i - t * F;
    const float g = ldf(gate, t * ldg + c);
    const float s = 1.f / (1.f + expf(-g));
    stf(out, i, ldf(y, t * ldy + c) * (kind == 1 ? g * s : s));
  }
}

// kinds: 0 gelu_tanh(g) * u, 1 g' * sigmoid(alpha g') * (u' + 1) with g' = min(g, limit), u' = clamp(u, +-limit)
// (limit <= 0: no clamp), 5 relu(g) * u -- these read [T, 2F] = [gate | up]; 2 tanh, 3 silu, 4 erf-gelu,
// 6 limit * tanh(x / limit), 7 relu(x)^2: elementwise on [T, F].
// Elementwise kinds take a factor per row: logical row i is row row_map[i] (or i) and its input is multiplied by
// row_scale[i] before the function (experts whose router weight scales their input).  Gated kinds take a bias [2F]
// that is added to [gate | up] first.
__device__ __forceinline__ float act_elem(float v, int kind, float limit) {
  return kind == 2   ? tanhf(v)
         : kind == 3 ? v / (1.f + expf(-v))
         : kind == 4 ? 0.5f * v * (1.f + erff(v * 0.7071067811865476f))
         : kind == 7 ? (v > 0.f ? v * v : 0.f)
                     : limit * tanhf(v / limit);
}
// The gated kinds on one pair (g, u).
__device__ __forceinline__ float act_pair(float g, float u, int kind, float limit, float alpha) {
  if (kind == 0) return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  if (kind == 5) return fmaxf(g, 0.f) * u;
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return g / (1.f + expf(-alpha * g)) * (u + 1.f);
}
template <typename TA>
__global__ void act_kernel(TA* __restrict__ out, const TA* __restrict__ x, int T, int F, int kind, float limit,
                           float alpha, const float* __restrict__ row_scale, const int* __restrict__ row_map,
                           const TA* __restrict__ bias) {
  const size_t n = (size_t)T * F;
  if (kind >= 2 && kind != 5 && row_scale == nullptr && row_map == nullptr && n % 4 == 0 &&
      ((uintptr_t)x | (uintptr_t)out) % (4 * sizeof(TA)) == 0) {   // no row index needed
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n / 4; i += (size_t)gridDim.x * blockDim.x) {
      f32x4 v = ldf4(x + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = act_elem(v[e], kind, limit);
      stf4(out + 4 * i, v);
    }
    return;
  }
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const size_t t = i / F, c = i - t * F;
    float y;
    size_t o = i;
    if (kind >= 2 && kind != 5) {
      if (row_map != nullptr) o = (size_t)row_map[t] * F + c;
      float v = ldf(x, o);
      if (row_scale != nullptr) v *= row_scale[t];
      y = act_elem(v, kind, limit);
    } else {
      float g = ldf(x, t * 2 * F + c), u = ldf(x, t * 2 * F + F + c);
      if (bias != nullptr) {
        g += ldf(bias, c);
        u += ldf(bias, F + c);
      }
      y = act_pair(g, u, kind, limit, alpha);
    }
    stf(out, o, y);
  }
}
// The gated kinds on rows of whole vectors (F % 4 == 0, aligned pointers): blocks (slice of the row, rows in turn).
template <typename TA>
__global__ __launch_bounds__(256) void act_gated_kernel(TA* __restrict__ out, const TA* __restrict__ x, int T, int F,
                                                        int kind, float limit, float alpha,
                                                        const TA* __restrict__ bias) {
  const int c = 4 * (blockIdx.x * 256 + threadIdx.x);
  if (c >= F) return;
  f32x4 bg = f32x4{0.f, 0.f, 0.f, 0.f}, bu = bg;
  if (bias != nullptr) {
    bg = ldf4(bias + c);
    bu = ldf4(bias + F + c);
  }
  for (int t = blockIdx.y; t < T; t += gridDim.y) {
    const f32x4 g = ldf4(x + (size_t)t * 2 * F + c), u = ldf4(x + (size_t)t * 2 * F + F + c);
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = act_pair(g[e] + bg[e], u[e] + bu[e], kind, limit, alpha);
    stf4(out + (size_t)t * F + c, y);
  }
}

// out[t] = ca * a[t] / rms(a[t]) * wa + cb * b[t] / rms(b[t]) * wb (b optional): the outputs of two mixers that run side
// by side, each normed over the row in fp32, joined.  One workgroup per row.  `lda`: the row stride of a (a view into a
// wider projection).  groups > 1 (a alone): every one of that many equal consecutive parts of the row is divided by its
// own root mean square, one wave per part.  `gate` (optional, output type, row stride ldg): every element of the result
// times sigmoid(gate) (gkind 0) or silu(gate) (gkind 1).
template <typename TO>
__device__ __forceinline__ float gate_of(const TO* gate, size_t i, int gkind) {
  const float g = ldf(gate, i), s = 1.f / (1.f + expf(-g));
  return gkind == 1 ? g * s : s;
}
// The single-input form without groups for rows of whole vectors (W % 4 == 0, W <= 1024 NV, every pointer and stride
// aligned to four elements): all loads ahead of the reduction, everything in registers.
template <typename TA, typename TO, int NV>
__global__ __launch_bounds__(256) void norm_row_kernel(TO* __restrict__ out, const TA* __restrict__ a, long lda,
                                                       const TA* __restrict__ wa, float eps, float ca, int W,
                                                       const TO* __restrict__ gate, long ldg, int gkind) {
  __shared__ float red[16];
  const TA* ar = a + (size_t)blockIdx.x * lda;
  const TO* gr = gate != nullptr ? gate + (size_t)blockIdx.x * ldg : nullptr;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 v[NV], wv[NV], gv[NV];
  float ss = 0.f;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int i = 4 * (threadIdx.x + 256 * n);
    const bool in = i < W;
    v[n] = in ? ldf4(ar + i) : zero;
    wv[n] = in ? ldf4(wa + i) : zero;
    gv[n] = in && gr != nullptr ? ldf4(gr + i) : zero;
  }
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += v[n][e] * v[n][e];
  ss = row_total(ss, red + 8);
  const float inv = ca / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int i = 4 * (threadIdx.x + 256 * n);
    if (i >= W) continue;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = v[n][e] * inv * wv[n][e];
      if (gr != nullptr) {
        const float s = 1.f / (1.f + expf(-gv[n][e]));
        y[e] *= gkind == 1 ? gv[n][e] * s : s;
      }
    }
    stf4(out + (size_t)blockIdx.x * W + i, y);
  }
}

template <typename TA, typename TO>
__global__ __launch_bounds__(256) void norm_mix_kernel(TO* __restrict__ out, const TA* __restrict__ a, long lda,
                                                       const TA* __restrict__ wa, const TA* __restrict__ b,
                                                       const TA* __restrict__ wb, float eps, float ca, float cb, int W,
                                                       int groups, const TO* __restrict__ gate, long ldg, int gkind) {
  __shared__ float red[16];
  const size_t base = (size_t)blockIdx.x * W;
  const TA* ar = a + (size_t)blockIdx.x * lda;
  if (groups > 1) {
    const int Wg = W / groups, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    for (int g = wave; g < groups; g += nw) {
      const size_t o = (size_t)g * Wg;
      float sg = 0.f;
      for (int i = lane; i < Wg; i += 64) {
        const float v = ldf(ar, o + i);
        sg += v * v;
      }
      sg = wave_sum(sg);
      const float inv = ca / sqrtf(sg / (float)Wg + eps);
      for (int i = lane; i < Wg; i += 64) {
        const float y = ldf(ar, o + i) * inv * ldf(wa, o + i);
        stf(out, base + o + i, gate != nullptr ? y * gate_of(gate, (size_t)blockIdx.x * ldg + o + i, gkind) : y);
      }
    }
    return;
  }
  float sa = 0.f, sb = 0.f;
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const float va = ldf(ar, i);
    sa += va * va;
    if (b != nullptr) {
      const float vb = ldf(b, base + i);
      sb += vb * vb;
    }
  }
  sa = block_sum(sa, red);
  const float ia = ca / sqrtf(sa / (float)W + eps);
  float ib = 0.f;
  if (b != nullptr) {   // uniform branch
    sb = block_sum(sb, red);
    ib = cb / sqrtf(sb / (float)W + eps);
  }
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    float y = ldf(ar, i) * ia * ldf(wa, i);
    if (b != nullptr) y += ldf(b, base + i) * ib * ldf(wb, i);
    if (gate != nullptr) y *= gate_of(gate, (size_t)blockIdx.x * ldg + i, gkind);
    stf(out, base + i, y);
  }
}

// C = A W^T for any M, N, K and any row strides: 64 x 64 output tile per workgroup, 16-deep k steps staged through LDS
// as fp32, 4 x 4 outputs per thread, fp32 FMA accumulation in k order (a row's result does not depend on which rows
// share its tile).  Three forms:
//   plain / strided-batched: blockIdx.z = batch g, operands offset by g * (sA, sW, sC);
//   row gather: A row r is A[a_rows[r]];
//   grouped: tiles[y] = (group, first row, rows) lists the row tiles of variable-size groups over one compact row
//   space (a mixture-of-experts' sorted tokens); group g uses W + g * sW; tiles with group < 0 are padding.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void gemm_any_kernel(TO* __restrict__ C, const TI* __restrict__ A,
                                                       const TI* __restrict__ Wt, int M, int N, int K, long lda,
                                                       long ldw, long ldc, long sA, long sW, long sC,
                                                       const int* __restrict__ a_rows, const int* __restrict__ tiles) {
  constexpr int BM = 64, BN = 64, BK = 16, LD = BM + 4;
  __shared__ __attribute__((aligned(16))) float As[BK][LD];
  __shared__ __attribute__((aligned(16))) float Ws[BK][LD];
  int row0, rows;
  if (tiles != nullptr) {
    const int g = tiles[3 * blockIdx.y];
    if (g < 0) return;
    row0 = tiles[3 * blockIdx.y + 1];
    rows = tiles[3 * blockIdx.y + 2];
    Wt += (size_t)g * sW;
  } else {
    row0 = blockIdx.y * BM;
    rows = min(BM, M - row0);
    A += (size_t)blockIdx.z * sA;
    Wt += (size_t)blockIdx.z * sW;
    C += (size_t)blockIdx.z * sC;
  }
  const int col0 = blockIdx.x * BN;
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int kk = tid & 15, r_l = tid >> 4;          // loader: k index, first of 4 rows (r_l + 16 i)
  size_t a_off[4], w_off[4];
  bool a_ok[4], w_ok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r_l + 16 * i;
    a_ok[i] = r < rows;
    const int gr = a_ok[i] ? (a_rows != nullptr ? a_rows[row0 + r] : row0 + r) : 0;
    a_off[i] = (size_t)gr * lda;
    w_ok[i] = col0 + r < N;
    w_off[i] = (size_t)(w_ok[i] ? col0 + r : 0) * ldw;
  }
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += BK) {
    const bool kin = k0 + kk < K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      As[kk][r_l + 16 * i] = (kin && a_ok[i]) ? ldf(A, a_off[i] + k0 + kk) : 0.f;
      Ws[kk][r_l + 16 * i] = (kin && w_ok[i]) ? ldf(Wt, w_off[i] + k0 + kk) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(&As[k][ty * 4]);
      const f32x4 b = *reinterpret_cast<const f32x4*>(&Ws[k][tx * 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = ty * 4 + i;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = col0 + tx * 4 + j;
      if (c < N) stf(C, (size_t)(row0 + r) * ldc + c, acc[i][j]);
    }
  }
}

// The same product for fp32 operands whose rows are 16-byte aligned (k and every stride a multiple of 4 elements) on the
// matrix cores' fp32 instruction (v_mfma_f32_32x32x2_f32: fp32 products and sums, nothing rounded in between).  A workgroup
// of 8 waves owns a 32 x (32 NN) output tile, in the swapped orientation C^T = W A^T; its waves share k instead of the tile:
// of every 64-deep step, staged through two LDS buffers, wave w multiplies the elements [8 w, 8 w + 8), so small tiles still
// give every SIMD two waves.  A lane reads 4 consecutive k of its row and spends one on each of 4 instructions.  PF steps'
// loads are in flight.  The waves' sums meet in LDS in wave order: an output's accumulation order depends on K alone, not on
// the tile or the rows that share it.  Same three forms.
// It takes what k8s_gemm_f32_parts_rule and k8s_gemm_f32_rule leave it: few rows, few tiles, short listed groups, depths below 512 or no multiple of 32; the rest
// runs on gemm_f32.hip's tiles.  Bound by the loads of weights that no other workgroup reads (16 rows, from memory: 2048 x 2048
// (N x K) 19.6 us, 4096 x 14336 120 us), and with many rows by the fp32 matrix rate (157 TFLOP/s; a 32 x 32 x 2048 tile is 7 us of
// a CU's four pipes).
template <typename TO, int NN>
__global__ __launch_bounds__(512) void gemm_f32_kernel(TO* __restrict__ C, const float* __restrict__ A,
                                                       const float* __restrict__ Wt, int M, int N, int K, long lda,
                                                       long ldw, long ldc, long sA, long sW, long sC,
                                                       const int* __restrict__ a_rows, const int* __restrict__ tiles) {
  typedef float f32x16 __attribute__((ext_vector_type(16)));
  constexpr int BM = 32, BN = 32 * NN, BK = 64, LD = BK + 4, PF = 4, PER = 64 / BM;
  constexpr int STAGE = (BM + BN) * LD;            // floats of one LDS buffer: A rows, then W rows
  constexpr int LDS = 2 * STAGE > 8 * 16 * 64 ? 2 * STAGE : 8 * 16 * 64;
  __shared__ __attribute__((aligned(16))) float sm[LDS];
  int row0, rows;
  if (tiles != nullptr) {                          // PER blocks per listed tile of at most 64 rows
    const int y = blockIdx.y / PER, sub = (blockIdx.y - y * PER) * BM;
    const int g = tiles[3 * y];
    if (g < 0) return;
    row0 = tiles[3 * y + 1] + sub;
    rows = min(BM, tiles[3 * y + 2] - sub);
    if (rows <= 0) return;
    Wt += (size_t)g * sW;
  } else {
    row0 = blockIdx.y * BM;
    rows = min(BM, M - row0);
    A += (size_t)blockIdx.z * sA;
    Wt += (size_t)blockIdx.z * sW;
    C += (size_t)blockIdx.z * sC;
  }
  const int col0 = blockIdx.x * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 31, h = lane >> 5;
  const int lr = tid >> 4, lc = 4 * (tid & 15);    // loader: row lr (W: + 32 b), 4 elements from lc of the step
  // rows and columns past the end repeat the last one (they are not stored)
  const int ar = row0 + min(lr, rows - 1);
  const float* ap = A + (size_t)(a_rows != nullptr ? a_rows[ar] : ar) * lda;
  const float* wp[NN];
#pragma unroll
  for (int b = 0; b < NN; ++b) wp[b] = Wt + (size_t)min(col0 + 32 * b + lr, N - 1) * ldw;
  f32x4 ra[PF], rw[PF][NN];
  auto fetch = [&](f32x4& fa, f32x4 (&fw)[NN], int k0) {     // past the end: the row's last elements, staged as zeros
    const int k = min(k0 + lc, K - 4);
    fa = *reinterpret_cast<const f32x4*>(ap + k);
#pragma unroll
    for (int b = 0; b < NN; ++b) fw[b] = *reinterpret_cast<const f32x4*>(wp[b] + k);
  };
  f32x16 acc[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[n][i] = 0.f;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < PF; ++p) fetch(ra[p], rw[p], BK * p);
  for (int k0 = 0; k0 < K; k0 += BK * PF) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int k = k0 + BK * p;
      if (k >= K) break;                           // uniform
      float* st = sm + (p & 1) * STAGE;
      const bool in = k + lc < K;
      *reinterpret_cast<f32x4*>(st + lr * LD + lc) = in ? ra[p] : zero;
#pragma unroll
      for (int b = 0; b < NN; ++b) *reinterpret_cast<f32x4*>(st + (BM + 32 * b + lr) * LD + lc) = in ? rw[p][b] : zero;
      lds_barrier();         // this buffer is written; the other one was read before every wave came here
      fetch(ra[p], rw[p], k + BK * PF);
      const f32x4 fa = *reinterpret_cast<const f32x4*>(st + li * LD + 8 * wave + 4 * h);
      f32x4 fw[NN];
#pragma unroll
      for (int b = 0; b < NN; ++b) fw[b] = *reinterpret_cast<const f32x4*>(st + (BM + 32 * b + li) * LD + 8 * wave + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NN; ++n) acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[n][i], fa[i], acc[n], 0, 0, 0);
    }
  }
  // acc[n][4 q + i] = C[row li][col 32 n + 8 q + 4 h + i], this wave's share of k
  float(*red)[16][64] = reinterpret_cast<float(*)[16][64]>(sm);
#pragma unroll
  for (int n = 0; n < NN; ++n) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) red[wave][i][lane] = acc[n][i];
    __syncthreads();
    float y[2] = {0.f, 0.f};                       // thread (wave, lane) finishes the elements 2 wave, 2 wave + 1
#pragma unroll
    for (int v = 0; v < 8; ++v)
#pragma unroll
      for (int e = 0; e < 2; ++e) y[e] += red[v][2 * wave + e][lane];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int x = 2 * wave + e, c = col0 + 32 * n + 8 * (x >> 2) + 4 * h + (x & 3);
      if (li < rows && c < N) stf(C, (size_t)(row0 + li) * ldc + c, y[e]);
    }
  }
}

// The same product for bf16 operands whose rows are 16-byte aligned (k and every stride a multiple of 8 elements) on
// the matrix cores: 64 x 64 or (many rows and columns) 64 x 128 output tile, 32-deep k steps, 4 waves of 32 x 32 or
// 32 x 64 (2 x NF v_mfma_f32_16x16x32_bf16) in the swapped orientation C^T = W A^T, so a lane ends with 4 consecutive
// columns of one row; an output's accumulation is the same in both tile shapes.  The next k step's global
// loads are in flight during the current step's MFMAs.  Same three forms (batched, row gather, grouped tiles); the
// accumulation order of an output does not depend on M or on the rows that share its tile.
template <typename TO, int NF>   // NF 16-column fragments per wave: output tile 64 x (32 NF)
__global__ __launch_bounds__(256) void gemm_mfma_kernel(TO* __restrict__ C, const bf16_t* __restrict__ A,
                                                        const bf16_t* __restrict__ Wt, int M, int N, int K, long lda,
                                                        long ldw, long ldc, long sA, long sW, long sC,
                                                        const int* __restrict__ a_rows, const int* __restrict__ tiles) {
  constexpr int BM = 64, BN = 32 * NF, BK = 32, LDK = BK + 8;   // rows of 80 bytes: 16-byte aligned fragments
  constexpr int WL = BN / 64;                                    // W rows per loader thread
  __shared__ __attribute__((aligned(16))) bf16_t As[BM][LDK];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[BN][LDK];
  int row0, rows;
  if (tiles != nullptr) {
    const int g = tiles[3 * blockIdx.y];
    if (g < 0) return;
    row0 = tiles[3 * blockIdx.y + 1];
    rows = tiles[3 * blockIdx.y + 2];
    Wt += (size_t)g * sW;
  } else {
    row0 = blockIdx.y * BM;
    rows = min(BM, M - row0);
    A += (size_t)blockIdx.z * sA;
    Wt += (size_t)blockIdx.z * sW;
    C += (size_t)blockIdx.z * sC;
  }
  const int col0 = blockIdx.x * BN;
  const int tid = threadIdx.x;
  // loader: thread -> (row tid / 4 (+ 64 c for W), 8-element chunk tid % 4)
  const int lr = tid >> 2, lc = tid & 3;
  const bool a_ok = lr < rows;
  const int gr = a_ok ? (a_rows != nullptr ? a_rows[row0 + lr] : row0 + lr) : 0;
  const bf16_t* ap = A + (size_t)gr * lda + lc * 8;
  const bf16_t* wp[WL];
  bool w_ok[WL];
#pragma unroll
  for (int c = 0; c < WL; ++c) {
    w_ok[c] = col0 + lr + 64 * c < N;
    wp[c] = Wt + (size_t)(w_ok[c] ? col0 + lr + 64 * c : 0) * ldw + lc * 8;
  }
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  u32x4 ra, rw[WL];
  auto fetch = [&](int k0) {
    const bool kin = k0 + lc * 8 < K;
    ra = (kin && a_ok) ? *reinterpret_cast<const u32x4*>(ap + k0) : zero;
#pragma unroll
    for (int c = 0; c < WL; ++c) rw[c] = (kin && w_ok[c]) ? *reinterpret_cast<const u32x4*>(wp[c] + k0) : zero;
  };
  const int lane = tid & 63, wave = tid >> 6, li = lane & 15, g = lane >> 4;
  const int m0 = (wave & 1) * 32, n0 = (wave >> 1) * (16 * NF);
  f32x4 acc[NF][2];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[f][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    __syncthreads();
    *reinterpret_cast<u32x4*>(&As[lr][lc * 8]) = ra;
#pragma unroll
    for (int c = 0; c < WL; ++c) *reinterpret_cast<u32x4*>(&Ws[lr + 64 * c][lc * 8]) = rw[c];
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);
    bf16x8 wf[NF], af[2];
#pragma unroll
    for (int f = 0; f < NF; ++f) wf[f] = *reinterpret_cast<const bf16x8*>(&Ws[n0 + 16 * f + li][8 * g]);
#pragma unroll
    for (int j = 0; j < 2; ++j) af[j] = *reinterpret_cast<const bf16x8*>(&As[m0 + 16 * j + li][8 * g]);
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[f][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f], af[j], acc[f][j], 0, 0, 0);
  }
  // acc[f][j][i] = C[row m0 + 16 j + li][col n0 + 16 f + 4 g + i]
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = m0 + 16 * j + li;
    if (r >= rows) continue;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = col0 + n0 + 16 * f + 4 * g + i;
        if (c < N) stf(C, (size_t)(row0 + r) * ldc + c, acc[f][j][i]);
      }
  }
}

// An activation in the epilogue of the few-row products: elementwise (plain ones), or gated (grouped ones; weight rows [0, N)
// gate, [N, 2 N) up); the sums are not rounded ahead of it.  Gate / up of 8 experts of 2 x 2048 x 2048, 64 / 96 rows: 36.9 /
// 40.6 us with the launch behind it, 33.2 / 34.8 us; 8 x 128 x 2048 with tanh: 7.1 us, 5.6 us.
enum { FEW_NONE = 0, FEW_ELEM = 1, FEW_PAIR = 2 };
struct FewAct {
  int kind;
  float limit, alpha;
  int last;            // grouped: this group's limit is last_limit
  float last_limit;
};
// Grouped products of few rows (decoding with experts): a workgroup takes 16 columns of one row tile (at most 64 rows).  The
// weights go from memory straight into MFMA operands, no LDS staging; its 4 waves share the k range in 64-deep pieces (wave w
// the pieces w, w + 4, ...), several pieces' loads in flight each, and their sums meet in LDS.  Orientation as above, C^T =
// W A^T.  K % 64 == 0, rows 16-byte aligned.  NB row blocks of 16 (1: tiles of at most 16 rows; 4: any).
template <typename TO, int NB, int ACT>
__device__ __forceinline__ void gemm_group_tile(TO* C, const bf16_t* A, const bf16_t* Wt, int N, int K, long lda, long ldw,
                                                long ldc, const int* a_rows, int row0, int rows, float* red,
                                                const FewAct& act) {
  constexpr int U = NB == 1 ? 4 : 2;           // pieces in flight
  constexpr int NP = ACT == FEW_PAIR ? 2 : 1;  // weight rows of an output column: gate and up
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g4 = lane >> 4;
  const int col0 = blockIdx.x * 16;
  const bf16_t* wp[NP];
#pragma unroll
  for (int x = 0; x < NP; ++x) wp[x] = Wt + (size_t)(min(col0 + li, N - 1) + x * N) * ldw + 8 * g4;
  const bf16_t* ap[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int r = min(16 * b + li, rows - 1);
    ap[b] = A + (size_t)(a_rows != nullptr ? a_rows[row0 + r] : row0 + r) * lda + 8 * g4;
  }
  f32x4 acc[NP][NB];
#pragma unroll
  for (int x = 0; x < NP; ++x)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[x][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int pieces = K / 64;
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  for (int s0 = wave; s0 < pieces; s0 += 4 * U) {
    u32x4 wv[U][NP][2], av[U][NB][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + 4 * u;
      const bool in = s < pieces;              // uniform over the wave
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int x = 0; x < NP; ++x)
          wv[u][x][h] = in ? *reinterpret_cast<const u32x4*>(wp[x] + 64 * s + 32 * h) : zero;
#pragma unroll
        for (int b = 0; b < NB; ++b)
          av[u][b][h] = in && (NB == 1 || 16 * b < rows) ? *reinterpret_cast<const u32x4*>(ap[b] + 64 * s + 32 * h) : zero;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int x = 0; x < NP; ++x)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            acc[x][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[u][x][h]),
                                                                __builtin_bit_cast(bf16x8, av[u][b][h]), acc[x][b], 0, 0, 0);
  }
  // acc[x][b][i] = C[row 16 b + li][col col0 + 4 g4 + i], this wave's share of k
#pragma unroll
  for (int x = 0; x < NP; ++x)
#pragma unroll
    for (int b = 0; b < NB; ++b)
      *reinterpret_cast<f32x4*>(red + ((size_t)((wave * NP + x) * NB + b) * 64 + lane) * 4) = acc[x][b];
  __syncthreads();
  for (int b = wave; b < NB; b += 4) {
    const int r = 16 * b + li;
    if (r >= rows) continue;
    f32x4 y[NP];
#pragma unroll
    for (int x = 0; x < NP; ++x) {
      y[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(red + ((size_t)((w * NP + x) * NB + b) * 64 + lane) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[x][e] += v[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = col0 + 4 * g4 + e;
      if (c >= N) continue;
      float v = y[0][e];
      if constexpr (ACT == FEW_ELEM) v = act_elem(v, act.kind, act.limit);
      if constexpr (ACT == FEW_PAIR) v = act_pair(v, y[NP - 1][e], act.kind, act.limit, act.alpha);
      stf(C, (size_t)(row0 + r) * ldc + c, v);
    }
  }
}
template <typename TO, int ACT>
__global__ __launch_bounds__(256) void gemm_group_kernel(TO* __restrict__ C, const bf16_t* __restrict__ A,
                                                         const bf16_t* __restrict__ Wt, int N, int K, long lda, long ldw,
                                                         long ldc, long sW, const int* __restrict__ a_rows,
                                                         const int* __restrict__ tiles, FewAct act) {
  __shared__ __attribute__((aligned(16))) float red[(ACT == FEW_PAIR ? 2 : 1) * 4 * 4 * 64 * 4];
  const int g = tiles[3 * blockIdx.y];
  if (g < 0) return;
  const int row0 = tiles[3 * blockIdx.y + 1], rows = tiles[3 * blockIdx.y + 2];
  Wt += (size_t)g * sW;
  if (ACT == FEW_PAIR && g == act.last) act.limit = act.last_limit;
  if (rows <= 16) gemm_group_tile<TO, 1, ACT>(C, A, Wt, N, K, lda, ldw, ldc, a_rows, row0, rows, red, act);
  else gemm_group_tile<TO, 4, ACT>(C, A, Wt, N, K, lda, ldw, ldc, a_rows, row0, rows, red, act);
}

// The same for plain and strided-batched products whose 64 x 64 tiles would leave most of the chip idle (few rows, or few
// columns): workgroups (16 columns, 64 rows, batch).
template <typename TO, int ACT>
__global__ __launch_bounds__(256) void gemm_narrow_kernel(TO* __restrict__ C, const bf16_t* __restrict__ A,
                                                          const bf16_t* __restrict__ Wt, int M, int N, int K, long lda,
                                                          long ldw, long ldc, long sA, long sW, long sC, FewAct act) {
  __shared__ __attribute__((aligned(16))) float red[4 * 4 * 64 * 4];
  const int row0 = blockIdx.y * 64, rows = min(64, M - row0);
  A += (size_t)blockIdx.z * sA;
  Wt += (size_t)blockIdx.z * sW;
  C += (size_t)blockIdx.z * sC;
  if (rows <= 16) gemm_group_tile<TO, 1, ACT>(C, A, Wt, N, K, lda, ldw, ldc, nullptr, row0, rows, red, act);
  else gemm_group_tile<TO, 4, ACT>(C, A, Wt, N, K, lda, ldw, ldc, nullptr, row0, rows, red, act);
}

// A decode step's latent attention up to the attention itself, one launch for two: the tokens' cache rows and query rotation (plane 0),
// and the queries' unrotated parts taken into the latent space, gemm_narrow_kernel's work for a head a plane.  Neither reads what the
// other writes.
template <bool IL>
__global__ __launch_bounds__(256) void latent_begin_kernel(LatentRows<bf16_t> a, int T, bf16_t* __restrict__ q_abs,
                                                           const bf16_t* __restrict__ uk) {
  __shared__ __attribute__((aligned(16))) float red[4 * 4 * 64 * 4];
  if (blockIdx.z == 0) {
    for (int t = blockIdx.x; t < T; t += gridDim.x) {
      latent_row<bf16_t, IL>(a, t, red);
      __syncthreads();                             // the sums of the row before have been read
    }
    return;
  }
  const int h = blockIdx.z - 1;
  const bf16_t* A = a.q + (size_t)h * (a.Dn + a.R);
  const bf16_t* W = uk + (size_t)h * a.C * a.Dn;
  const long lda = (long)a.H * (a.Dn + a.R), ldc = (long)a.H * a.C;
  if (T <= 16) gemm_group_tile<bf16_t, 1, FEW_NONE>(q_abs + (size_t)h * a.C, A, W, a.C, a.Dn, lda, a.Dn, ldc, nullptr, 0, T, red, FewAct{});
  else gemm_group_tile<bf16_t, 4, FEW_NONE>(q_abs + (size_t)h * a.C, A, W, a.C, a.Dn, lda, a.Dn, ldc, nullptr, 0, T, red, FewAct{});
}

}  // namespace k8sllm

using namespace k8sllm;

// q_abs [T][H][C] = q's unrotated parts times uk [H][C][Dn]^T, and latent_kv_write, of bf16.  -5: a size or an alignment that this form
// does not take; nothing was launched.
extern "C" int k8s_latent_begin(void* q_abs, const void* uk, void* cache, const void* dkv, const void* normw, void* q, const float* cos_sin,
                                const int* positions, const int* slot_mapping, int T, int C, int R, int H, int Dn, int dims, float eps,
                                long ldd, int interleaved, hipStream_t s) {
  if (T <= 0) return 0;
  if (C <= 0 || R < 0 || dims < 0 || dims > R || (dims & 1) || H <= 0 || Dn <= 0 || ldd < C + R || !q_abs || !uk) return -1;
  const LatentRows<bf16_t> a = {(bf16_t*)cache, (const bf16_t*)dkv, (const bf16_t*)normw, (bf16_t*)q, cos_sin, positions, slot_mapping,
                                C, R, H, Dn, dims, eps, ldd};
  if (T > 64 || H >= 65535 || Dn % 64 || (Dn + R) % 8 || C % 16 || ((uintptr_t)q | (uintptr_t)uk | (uintptr_t)q_abs) % 16 || !latent_row_ok(a))
    return -5;
  const dim3 grid(C / 16, 1, H + 1);
  if (interleaved) latent_begin_kernel<true><<<grid, 256, 0, s>>>(a, T, (bf16_t*)q_abs, (const bf16_t*)uk);
  else latent_begin_kernel<false><<<grid, 256, 0, s>>>(a, T, (bf16_t*)q_abs, (const bf16_t*)uk);
  return (int)hipGetLastError();
}

extern "C" int k8s_embed_rows(float* out, void* copy, const int* ids, const void* table, int T, int W, int vocab,
                              float scale, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || vocab <= 0) return -1;
  if (f32) embed_rows_kernel<float><<<T, 256, 0, s>>>(out, (float*)copy, ids, (const float*)table, W, vocab, scale);
  else embed_rows_kernel<bf16_t><<<T, 256, 0, s>>>(out, (bf16_t*)copy, ids, (const bf16_t*)table, W, vocab, scale);
  return (int)hipGetLastError();
}

// pos and slots [B], ar [B + 1]; block_tables [B, max_blocks]
extern "C" int k8s_decode_meta(int* pos, int* slots, int* ar, const int* ctx, const int* block_tables, int max_blocks,
                               int B, int bs, hipStream_t s) {
  if (B < 0 || max_blocks < 0 || bs <= 0) return -1;
  decode_meta_kernel<<<(B + 256) / 256, 256, 0, s>>>(pos, slots, ar, ctx, block_tables, max_blocks, B, bs);
  return (int)hipGetLastError();
}

extern "C" int k8s_embed_step(float* out, void* copy, const int* ids, const void* table, int W, int vocab, float scale, int f32, int* pos,
                              int* slots, int* ar, const int* ctx, const int* block_tables, int max_blocks, int B, int bs,
                              hipStream_t s) {
  if (B <= 0 || max_blocks < 0 || bs <= 0 || W <= 0 || vocab <= 0) return -1;
  const int grid = B + (B + 256) / 256;
  if (f32) embed_step_kernel<float><<<grid, 256, 0, s>>>(out, (float*)copy, ids, (const float*)table, W, vocab, scale, pos, slots, ar, ctx,
                                                         block_tables, max_blocks, B, bs);
  else embed_step_kernel<bf16_t><<<grid, 256, 0, s>>>(out, (bf16_t*)copy, ids, (const bf16_t*)table, W, vocab, scale, pos, slots, ar, ctx,
                                                      block_tables, max_blocks, B, bs);
  return (int)hipGetLastError();
}

extern "C" int k8s_resnorm(float* x, const void* branch, const void* branch2, float mult, const void* rowvec,
                           const void* w, float offset, float eps, void* out, int T, int W, int groups, int f32,
                           hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || (w != nullptr && out == nullptr) || groups < 1 || W % groups || (branch2 != nullptr && branch == nullptr))
    return -1;
#define K8S_RN(TA, NV)                                                                                              \
  resnorm_row_kernel<TA, NV><<<T, 256, 0, s>>>(x, (const TA*)branch, (const TA*)branch2, mult, (const TA*)rowvec,     \
                                               (const TA*)w, offset, eps, (TA*)out, W)
#define K8S_RN_T(TA)                                                                                                \
  do {                                                                                                              \
    const bool vec = w != nullptr && groups == 1 && W % 4 == 0 && W <= 8192 && (uintptr_t)x % 16 == 0 &&             \
                     ((uintptr_t)branch | (uintptr_t)branch2 | (uintptr_t)rowvec | (uintptr_t)w | (uintptr_t)out) %  \
                             (4 * sizeof(TA)) == 0;                                                                 \
    if (!vec)                                                                                                       \
      resnorm_kernel<TA><<<T, 256, 0, s>>>(x, (const TA*)branch, (const TA*)branch2, mult, (const TA*)rowvec,        \
                                           (const TA*)w, offset, eps, (TA*)out, W, groups);                         \
    else if (W <= 1024) K8S_RN(TA, 1);                                                                              \
    else if (W <= 2048) K8S_RN(TA, 2);                                                                              \
    else if (W <= 4096) K8S_RN(TA, 4);                                                                              \
    else K8S_RN(TA, 8);                                                                                             \
  } while (0)
  if (f32) K8S_RN_T(float);
  else K8S_RN_T(bf16_t);
#undef K8S_RN_T
#undef K8S_RN
  return (int)hipGetLastError();
}

// -5: a size or an alignment that this form does not take; nothing was launched
extern "C" int k8s_norm_shift(void* out, float* x, const void* branch, float mult, const void* rowvec, const void* w, float offset,
                              float eps, const void* mu, void* state, const int* seq_slots, const int* positions, int n, int T, int W,
                              int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || n <= 0 || w == nullptr || out == nullptr || state == nullptr || mu == nullptr) return -1;
  if (n > SHIFT_MIXES || W % 4 || W > 4096 || (uintptr_t)x % 16 ||
      ((uintptr_t)branch | (uintptr_t)rowvec | (uintptr_t)w | (uintptr_t)out | (uintptr_t)mu | (uintptr_t)state) % (f32 ? 16 : 8))
    return -5;
#define K8S_NS(TA, NV)                                                                                                       \
  norm_shift_kernel<TA, NV><<<T, 256, 0, s>>>((TA*)out, x, (const TA*)branch, mult, (const TA*)rowvec, (const TA*)w, offset, eps, \
                                              (const TA*)mu, (TA*)state, seq_slots, positions, n, T, W)
#define K8S_NS_T(TA)                   \
  do {                                 \
    if (W <= 1024) K8S_NS(TA, 1);      \
    else if (W <= 2048) K8S_NS(TA, 2); \
    else K8S_NS(TA, 4);                \
  } while (0)
  if (f32) K8S_NS_T(float);
  else K8S_NS_T(bf16_t);
#undef K8S_NS_T
#undef K8S_NS
  return (int)hipGetLastError();
}

extern "C" int k8s_norm_mix(void* out, const void* a, long lda, const void* wa, const void* b, const void* wb,
                            float eps, float ca, float cb, int T, int W, int groups, const void* gate, long ldg,
                            int gkind, int in_f32, int out_f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || a == nullptr || wa == nullptr || (b != nullptr && wb == nullptr) || lda < W) return -1;
  if (groups < 1 || W % groups || (groups > 1 && b != nullptr)) return -1;
  if (gate != nullptr && (ldg < W || gkind < 0 || gkind > 1)) return -1;
#define K8S_NM(TA, TO)                                                                                             \
  norm_mix_kernel<TA, TO><<<T, 256, 0, s>>>((TO*)out, (const TA*)a, lda, (const TA*)wa, (const TA*)b, (const TA*)wb, \
                                            eps, ca, cb, W, groups, (const TO*)gate, ldg, gkind)
#define K8S_NR(TA, TO, NV) \
  norm_row_kernel<TA, TO, NV><<<T, 256, 0, s>>>((TO*)out, (const TA*)a, lda, (const TA*)wa, eps, ca, W, (const TO*)gate, \
                                                ldg, gkind)
#define K8S_NM_T(TA, TO)                                                                              \
  do {                                                                                                \
    const bool vec = b == nullptr && groups == 1 && W % 4 == 0 && W <= 8192 && lda % 4 == 0 &&        \
                     (uintptr_t)a % (4 * sizeof(TA)) == 0 && (uintptr_t)wa % (4 * sizeof(TA)) == 0 && \
                     (uintptr_t)out % (4 * sizeof(TO)) == 0 && (uintptr_t)gate % (4 * sizeof(TO)) == 0 && ldg % 4 == 0; \
    if (!vec) K8S_NM(TA, TO);                                                                         \
    else if (W <= 1024) K8S_NR(TA, TO, 1);                                                            \
    else if (W <= 2048) K8S_NR(TA, TO, 2);                                                            \
    else if (W <= 4096) K8S_NR(TA, TO, 4);                                                            \
    else K8S_NR(TA, TO, 8);                                                                           \
  } while (0)
  if (in_f32 && out_f32) K8S_NM_T(float, float);
  else if (in_f32) K8S_NM_T(float, bf16_t);
  else if (out_f32) K8S_NM_T(bf16_t, float);
  else K8S_NM_T(bf16_t, bf16_t);
#undef K8S_NM_T
#undef K8S_NR
#undef K8S_NM
  return (int)hipGetLastError();
}

extern "C" int k8s_postnorm(float* x, const void* branch, const void* branch2, float alpha, float c1, float c2,
                            float gain, float eps, void* out, int T, int W, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || x == nullptr || (branch2 != nullptr && branch == nullptr)) return -1;
  if (f32)
    postnorm_kernel<float><<<T, 256, 0, s>>>(x, (const float*)branch, (const float*)branch2, alpha, c1, c2, gain, eps,
                                             (float*)out, W);
  else
    postnorm_kernel<bf16_t><<<T, 256, 0, s>>>(x, (const bf16_t*)branch, (const bf16_t*)branch2, alpha, c1, c2, gain,
                                              eps, (bf16_t*)out, W);
  return (int)hipGetLastError();
}

// branch_f32: the branch is fp32 whatever the activation type of w and out
extern "C" int k8s_branchnorm(float* x, const void* branch, const void* w, const void* bias, const void* nw, float gain,
                              const void* dotw, float* dot, float eps, void* out, int T, int W, int branch_f32, int f32,
                              hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || x == nullptr || (branch != nullptr && w == nullptr) || (f32 && !branch_f32)) return -1;
  if ((branch == nullptr && (bias != nullptr || nw == nullptr)) || (nw != nullptr && out == nullptr)) return -1;
  if (dot != nullptr && (nw == nullptr || dotw == nullptr)) return -1;
#define K8S_BN(TB, TA, NV)                                                                                               \
  branchnorm_kernel<TB, TA, NV><<<T, 256, 0, s>>>(x, (const TB*)branch, (const TA*)w, (const TA*)bias, (const TA*)nw, gain, \
                                                  (const TA*)dotw, dot, eps, (TA*)out, W, MoeBranch<TA>{})
#define K8S_BN_T(TB, TA)                                                                                                \
  do {                                                                                                                  \
    const bool vec = W % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)branch % (4 * sizeof(TB)) == 0 &&               \
                     ((uintptr_t)w | (uintptr_t)out | (uintptr_t)bias | (uintptr_t)nw | (uintptr_t)dotw) % (4 * sizeof(TA)) == 0; \
    if (!vec || W > 8192) K8S_BN(TB, TA, 0);                                                               \
    else if (W <= 1024) K8S_BN(TB, TA, 1);                                                                 \
    else if (W <= 2048) K8S_BN(TB, TA, 2);                                                                 \
    else if (W <= 4096) K8S_BN(TB, TA, 4);                                                                 \
    else K8S_BN(TB, TA, 8);                                                                                \
  } while (0)
  if (f32) K8S_BN_T(float, float);
  else if (branch_f32) K8S_BN_T(float, bf16_t);
  else K8S_BN_T(bf16_t, bf16_t);
#undef K8S_BN_T
#undef K8S_BN
  return (int)hipGetLastError();
}

// The same behind experts: the branch is their combine (MoeBranch), W % 4 == 0 up to 8192, every pointer aligned to four elements.
extern "C" int k8s_branchnorm_moe(float* x, const void* D, const int* pos, int cols, int top, float scale, const void* shared,
                                  const float* logits, int ld, const void* w, const void* nw, float gain, const void* dotw,
                                  float* dot, float eps, void* out, int T, int W, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (W <= 0 || W % 4 || W > 8192 || x == nullptr || D == nullptr || pos == nullptr || w == nullptr || top <= 0) return -1;
  if (cols != top && (cols != top + 1 || shared != nullptr)) return -1;
  if ((nw != nullptr && out == nullptr) || (dot != nullptr && (nw == nullptr || dotw == nullptr))) return -1;
  if ((uintptr_t)x % 16 || ((uintptr_t)D | (uintptr_t)shared | (uintptr_t)w | (uintptr_t)nw | (uintptr_t)dotw | (uintptr_t)out) % (f32 ? 16 : 8))
    return -1;
#define K8S_BM(TA, NV)                                                                                                      \
  branchnorm_kernel<TA, TA, NV, true><<<T, 256, 0, s>>>(x, (const TA*)nullptr, (const TA*)w, (const TA*)nullptr, (const TA*)nw, \
                                                        gain, (const TA*)dotw, dot, eps, (TA*)out, W,                        \
                                                        MoeBranch<TA>{(const TA*)D, pos, (const TA*)shared, logits, cols, top, ld, scale})
#define K8S_BM_T(TA)                                                                    \
  do {                                                                                  \
    if (W <= 1024) K8S_BM(TA, 1);                                                       \
    else if (W <= 2048) K8S_BM(TA, 2);                                                  \
    else if (W <= 4096) K8S_BM(TA, 4);                                                  \
    else K8S_BM(TA, 8);                                                                 \
  } while (0)
  if (f32) K8S_BM_T(float);
  else K8S_BM_T(bf16_t);
#undef K8S_BM_T
#undef K8S_BM
  return (int)hipGetLastError();
}

// y_f32: y is fp32 whatever the activation type (an fp32 intermediate gated into the activation type)
extern "C" int k8s_gate_mul(void* out, const void* y, long ldy, const void* gate, long ldg, int T, int F, int kind,
                            int y_f32, int f32, hipStream_t s) {
  if (T <= 0 || F <= 0) return 0;
  if (kind < 0 || kind > 1 || ldy < F || ldg < F || (f32 && !y_f32)) return -1;
  const size_t n = (size_t)T * F;
  const int blocks = (int)((n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256);
  if (f32)
    gate_mul_kernel<float, float><<<blocks, 256, 0, s>>>((float*)out, (const float*)y, ldy, (const float*)gate, ldg, T,
                                                         F, kind);
  else if (y_f32)
    gate_mul_kernel<float, bf16_t><<<blocks, 256, 0, s>>>((bf16_t*)out, (const float*)y, ldy, (const bf16_t*)gate, ldg,
                                                          T, F, kind);
  else
    gate_mul_kernel<bf16_t, bf16_t><<<blocks, 256, 0, s>>>((bf16_t*)out, (const bf16_t*)y, ldy, (const bf16_t*)gate,
                                                           ldg, T, F, kind);
  return (int)hipGetLastError();
}

extern "C" int k8s_act(void* out, const void* x, int T, int F, int kind, float limit, float alpha,
                       const float* row_scale, const int* row_map, const void* bias, int f32, hipStream_t s) {
  if (T <= 0 || F <= 0) return 0;
  const bool gated = kind < 2 || kind == 5;
  if (kind < 0 || kind > 7 || (gated && (row_scale != nullptr || row_map != nullptr)) || (kind == 6 && !(limit > 0.f)) ||
      (!gated && bias != nullptr))
    return -1;
  if (gated && F % 4 == 0 && ((uintptr_t)x | (uintptr_t)out | (uintptr_t)bias) % (f32 ? 16 : 8) == 0) {
    const int gx = (F / 4 + 255) / 256;
    const int rows = 8192 / gx < 1 ? 1 : 8192 / gx;
    const dim3 grid(gx, T < rows ? T : rows);
    if (f32) act_gated_kernel<float><<<grid, 256, 0, s>>>((float*)out, (const float*)x, T, F, kind, limit, alpha,
                                                          (const float*)bias);
    else act_gated_kernel<bf16_t><<<grid, 256, 0, s>>>((bf16_t*)out, (const bf16_t*)x, T, F, kind, limit, alpha,
                                                       (const bf16_t*)bias);
    return (int)hipGetLastError();
  }
  const size_t n = (size_t)T * F;
  const size_t nt = gated ? n : (n + 3) / 4;   // elementwise kinds: four elements per thread
  const int blocks = (int)((nt + 255) / 256 > 4096 ? 4096 : (nt + 255) / 256);
  if (f32) act_kernel<float><<<blocks, 256, 0, s>>>((float*)out, (const float*)x, T, F, kind, limit, alpha,
                                                    row_scale, row_map, (const float*)bias);
  else act_kernel<bf16_t><<<blocks, 256, 0, s>>>((bf16_t*)out, (const bf16_t*)x, T, F, kind, limit, alpha,
                                                row_scale, row_map, (const bf16_t*)bias);
  return (int)hipGetLastError();
}

// act(A W^T) in bf16 of few rows: elementwise of a plain product (tiles == nullptr; M rows), or a gated `kind` of a grouped one
// (tiles, W [groups, 2 N, K]; group `last`, if there is one, with last_limit).  K % 64 == 0, rows of whole 16-byte vectors.
extern "C" int k8s_gemm_few_act(void* C, const void* A, const void* W, int M, int N, int K, long lda, const int* a_rows,
                                const int* tiles, int ntiles, int kind, float limit, float alpha, int last, float last_limit,
                                hipStream_t s) {
  const bool pair = kind == 0 || kind == 1 || kind == 5;
  if (N <= 0 || K <= 0 || K % 64 || lda % 8 || kind < 0 || kind > 7 || (((uintptr_t)A | (uintptr_t)W) & 15)) return -1;
  if (pair != (tiles != nullptr) || (kind == 6 && !(limit > 0.f))) return -1;
  const int gy = pair ? ntiles : (M + 63) / 64;
  if (M <= 0 || gy <= 0) return 0;
  if (gy > 65535) return -2;
  const dim3 grid((N + 15) / 16, gy);
  const FewAct act{kind, limit, alpha, last, last_limit};
  if (pair)
    gemm_group_kernel<bf16_t, FEW_PAIR><<<grid, 256, 0, s>>>((bf16_t*)C, (const bf16_t*)A, (const bf16_t*)W, N, K, lda, K, N,
                                                             2L * N * K, a_rows, tiles, act);
  else
    gemm_narrow_kernel<bf16_t, FEW_ELEM><<<grid, 256, 0, s>>>((bf16_t*)C, (const bf16_t*)A, (const bf16_t*)W, M, N, K, lda, K,
                                                              N, 0, 0, 0, act);
  return (int)hipGetLastError();
}

extern "C" int k8s_gemm_f32_rule(int M, int N, int K, int batch, int ntiles);
extern "C" int k8s_gemm_f32_tiles(void* C, const float* A, const float* W, int M, int N, int K, long lda, long ldw, long ldc,
                                  int batch, long sA, long sW, long sC, const int* a_rows, const int* tiles, int ntiles,
                                  int out_f32, int fq, hipStream_t s);
extern "C" int k8s_gemm_f32_parts_rule(int M, int N, int K, int batch, int ntiles);
extern "C" int k8s_gemm_f32_parts(float* C, const float* A, const float* W, int M, int N, int K, long lda, long ldw, long ldc,
                                  int batch, long sA, long sW, long sC, const int* a_rows, const int* tiles, int ntiles, int tile,
                                  hipStream_t s);

extern "C" int k8s_gemm_any(void* C, const void* A, const void* W, int M, int N, int K, long lda, long ldw, long ldc,
                            int batch, long sA, long sW, long sC, const int* a_rows, const int* tiles, int ntiles,
                            int in_f32, int out_f32, hipStream_t s) {
  if (N <= 0 || K <= 0 || batch <= 0) return -1;
  int gy;
  if (tiles != nullptr) {
    if (ntiles <= 0) return 0;
    gy = ntiles;
    batch = 1;
  } else {
    if (M <= 0) return 0;
    gy = (M + 63) / 64;
  }
  if (gy > 65535 || batch > 65535) return -2;
  // bf16 rows that can be moved as 16-byte vectors: the bf16 MFMA kernels; fp32 ones: gemm_f32_parts.hip's tiles by its rule (fp32
  // outputs), else gemm_f32.hip's tiles or gemm_f32_kernel, by k8s_gemm_f32_rule; anything else: plain FMAs
  const bool vec = !in_f32 && K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0 && sA % 8 == 0 && sW % 8 == 0 &&
                   ((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0;
  if (vec && tiles != nullptr && K % 64 == 0 && M <= 32 * ntiles && M <= 512) {   // few rows per group
    const dim3 gg((N + 15) / 16, gy);
    if (out_f32) gemm_group_kernel<float, FEW_NONE><<<gg, 256, 0, s>>>((float*)C, (const bf16_t*)A, (const bf16_t*)W, N, K, lda, ldw,
                                                                       ldc, sW, a_rows, tiles, FewAct{});
    else gemm_group_kernel<bf16_t, FEW_NONE><<<gg, 256, 0, s>>>((bf16_t*)C, (const bf16_t*)A, (const bf16_t*)W, N, K, lda, ldw, ldc,
                                                                sW, a_rows, tiles, FewAct{});
    return (int)hipGetLastError();
  }
  // at most 128 tiles of 64 x 64: 16 columns per workgroup and k shared by its waves (8 x 128 x 2048: 26.8 us on two tiles,
  // 4.8 us; 2048 x 128 x 2048: 36 us on 64 tiles, 14.3 us; at 256 tiles both take the same)
  if (vec && tiles == nullptr && K % 64 == 0 && (long)gy * ((N + 63) / 64) * batch <= 128) {
    const dim3 gn((N + 15) / 16, gy, batch);
    if (out_f32) gemm_narrow_kernel<float, FEW_NONE><<<gn, 256, 0, s>>>((float*)C, (const bf16_t*)A, (const bf16_t*)W, M, N, K, lda,
                                                                        ldw, ldc, sA, sW, sC, FewAct{});
    else gemm_narrow_kernel<bf16_t, FEW_NONE><<<gn, 256, 0, s>>>((bf16_t*)C, (const bf16_t*)A, (const bf16_t*)W, M, N, K, lda, ldw,
                                                                 ldc, sA, sW, sC, FewAct{});
    return (int)hipGetLastError();
  }
  if (vec) {
    const bool wide = N >= 512 && (long)gy * ((N + 127) / 128) * batch >= 256;   // enough 64 x 128 tiles for the chip
    const dim3 g2((N + (wide ? 127 : 63)) / (wide ? 128 : 64), gy, batch);
#define K8S_GM(TO, NF) \
  gemm_mfma_kernel<TO, NF><<<g2, 256, 0, s>>>((TO*)C, (const bf16_t*)A, (const bf16_t*)W, M, N, K, lda, ldw, ldc, sA, \
                                              sW, sC, a_rows, tiles)
    if (out_f32) { if (wide) K8S_GM(float, 4); else K8S_GM(float, 2); }
    else { if (wide) K8S_GM(bf16_t, 4); else K8S_GM(bf16_t, 2); }
#undef K8S_GM
    return (int)hipGetLastError();
  }
  const dim3 grid((N + 63) / 64, gy, batch);
  const int gm = tiles != nullptr ? gy * 2 : (M + 31) / 32;     // fp32 tiles are 32 rows high
  if (in_f32 && K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && sA % 4 == 0 && sW % 4 == 0 && ((uintptr_t)A & 15) == 0 &&
      ((uintptr_t)W & 15) == 0 && gm <= 65535) {
    const int tile = out_f32 ? k8s_gemm_f32_parts_rule(M, N, K, batch, tiles != nullptr ? ntiles : 0) : 0;
    if (tile > 0) {
      const int rc = k8s_gemm_f32_parts((float*)C, (const float*)A, (const float*)W, M, N, K, lda, ldw, ldc, batch, sA, sW, sC, a_rows,
                                        tiles, ntiles, tile, s);
      if (rc != -2) return rc;
    }
    const int fq = k8s_gemm_f32_rule(M, N, K, batch, tiles != nullptr ? ntiles : 0);
    if (fq > 0) {
      const int rc = k8s_gemm_f32_tiles(C, (const float*)A, (const float*)W, M, N, K, lda, ldw, ldc, batch, sA, sW, sC, a_rows,
                                        tiles, ntiles, out_f32, fq, s);
      if (rc != -2) return rc;
    }
    // 32 x 64 tiles take about 1.8 times a 32 x 32 one (333 x 2048 x 2048: 50 us and 40 us; 512 rows: 49 and 52; 1 x 16384 x
    // 2048: 32 and 39): the shape whose tiles fill the last round over the CUs better
    const long t1 = (long)gm * ((N + 31) / 32) * batch, t2 = (long)gm * ((N + 63) / 64) * batch;
    const bool wide = 2.0 * (double)((t2 + 255) / 256) < 1.1 * (double)((t1 + 255) / 256);
    const dim3 gf((N + (wide ? 63 : 31)) / (wide ? 64 : 32), gm, batch);
#define K8S_GF(TO, NN) \
  gemm_f32_kernel<TO, NN><<<gf, 512, 0, s>>>((TO*)C, (const float*)A, (const float*)W, M, N, K, lda, ldw, ldc, sA, sW, sC, \
                                             a_rows, tiles)
    if (out_f32) { if (wide) K8S_GF(float, 2); else K8S_GF(float, 1); }
    else { if (wide) K8S_GF(bf16_t, 2); else K8S_GF(bf16_t, 1); }
#undef K8S_GF
    return (int)hipGetLastError();
  }
#define K8S_GA(TI, TO) \
  gemm_any_kernel<TI, TO><<<grid, 256, 0, s>>>((TO*)C, (const TI*)A, (const TI*)W, M, N, K, lda, ldw, ldc, sA, sW, sC, \
                                               a_rows, tiles)
  if (in_f32 && out_f32) K8S_GA(float, float);
  else if (in_f32) K8S_GA(float, bf16_t);
  else if (out_f32) K8S_GA(bf16_t, float);
  else K8S_GA(bf16_t, bf16_t);
#undef K8S_GA
  return (int)hipGetLastError();
}
