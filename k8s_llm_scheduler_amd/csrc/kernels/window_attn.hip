// Grouped-query sliding-window attention over a paged K / V cache, with pooled far context:
//   * the token at position p sees the cached tokens of positions max(0, p - window + 1) .. p and, beside them, one
//     key / value per block of P consecutive tokens that lies wholly before the window (block b = positions
//     b P .. b P + P - 1, seen when b P + P - 1 <= p - window): the mean of the block's cached keys / values;
//   * tokens and blocks share one softmax, optionally with a sink (a key of score 0 without a value: one more unit
//     in the denominator);
//   * instead of a window the mask can be chunked: positions are cut into chunks of `chunk` counted from 0 and a token
//     sees the tokens of its own chunk up to itself; scores can be soft-capped (cap tanh(s / cap)); the sink can be a
//     learned number per head (e^sink in the denominator); the output gate is per element or one number per head;
//   * a distance bias can be taken off the scores of the tokens: slope_h (p - j) for the key at position j (the sink has
//     none; it does not go with pooled blocks, which have no position of their own);
//   * queries and keys are prepared by one kernel per token: bias, optional RMS norm over the whole projection with a
//     weight, rotation of the first `dims` dimensions (interleaved pairs or the half layout), optional unit RMS per
//     head, value mixing with another layer's values, paged cache write (none for a layer that reads another's cache).
// Varlen batches as in mixers.hip: positions[t] < 0 marks an idle row that touches nothing.
#include "common.h"

namespace k8sllm {

// LDS written by some lanes of a wave is read by other lanes of the same wave: order the accesses.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One workgroup per token, one wave per head vector (H query heads, then G key heads; further passes when there are
// more vectors than waves).  x = proj + bias; (qnw / knw) x = x / rms(whole q or k projection) * weight;
// (x[2i], x[2i + 1]) -- half layout: (x[i], x[i + dims / 2]) -- turns by the angle of cos_sin[pos] = [cos(dims / 2) |
// sin(dims / 2)]; then x / sqrt(mean(x^2) + eps) when `unit`.  (hqw / hkw [D]) before the rotation every head is
// divided by its own root mean square and multiplied by the weight, the same for all heads.  Queries are written back
// in place, keys to
// kcache[slot][g][D].  Values: v = proj + bias, then (vfirst_in) v = (1 - lam) v + lam vfirst_in[t]; (vfirst_out)
// vfirst_out[t] = v in fp32; vcache[slot][g][V] = v.
template <typename TA>
__global__ __launch_bounds__(256) void window_kv_write_kernel(
    TA* __restrict__ kcache, TA* __restrict__ vcache, TA* __restrict__ qkv, long ld, int koff, int voff,
    const TA* __restrict__ qb, const TA* __restrict__ kb, const TA* __restrict__ vb, const float* __restrict__ cos_sin,
    const int* __restrict__ positions, const int* __restrict__ slot_mapping, const float* __restrict__ vfirst_in,
    float* __restrict__ vfirst_out, float lam, int H, int G, int D, int V, int dims, float eps, int unit,
    int half_layout, const TA* __restrict__ qnw, const TA* __restrict__ knw, const TA* __restrict__ hqw,
    const TA* __restrict__ hkw) {
  extern __shared__ float xs[];   // [waves][D]
  __shared__ float red[16];
  const int t = blockIdx.x;
  const int pos = positions[t];
  if (pos < 0) return;
  const int slot = slot_mapping[t];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, nw = blockDim.x >> 6;
  const int half = dims / 2;
  const float* cs = cos_sin + (size_t)pos * dims;
  TA* row = qkv + (size_t)t * ld;
  float* x = xs + (size_t)wave * D;
  float invq = 1.f, invk = 1.f;
  if (qnw != nullptr) {           // uniform branches: the norm runs over all heads of the projection at once
    float ss = 0.f;
    for (int i = tid; i < H * D; i += blockDim.x) {
      const float v = ldf(row, i) + (qb != nullptr ? ldf(qb, i) : 0.f);
      ss += v * v;
    }
    invq = 1.0f / sqrtf(block_sum(ss, red) / (float)(H * D) + eps);
  }
  if (knw != nullptr && G > 0) {
    float ss = 0.f;
    for (int i = tid; i < G * D; i += blockDim.x) {
      const float v = ldf(row + koff, i) + (kb != nullptr ? ldf(kb, i) : 0.f);
      ss += v * v;
    }
    invk = 1.0f / sqrtf(block_sum(ss, red) / (float)(G * D) + eps);
  }
  for (int hv = wave; hv < H + G; hv += nw) {
    const bool isq = hv < H;
    const int hd = isq ? hv : hv - H;
    const TA* src = row + (isq ? 0 : koff) + (size_t)hd * D;
    const TA* bias = isq ? qb : kb;
    const TA* nrm = isq ? qnw : knw;
    const TA* hnw = isq ? hqw : hkw;
    const float inv0 = isq ? invq : invk;
    float hs = 0.f;
    for (int d = lane; d < D; d += 64) {
      float v = ldf(src, d) + (bias != nullptr ? ldf(bias, (size_t)hd * D + d) : 0.f);
      if (nrm != nullptr) v *= inv0 * ldf(nrm, (size_t)hd * D + d);
      x[d] = v;
      hs += v * v;
    }
    if (hnw != nullptr) {            // uniform over the wave; every lane rescales the elements it wrote itself
      const float hinv = 1.0f / sqrtf(wave_sum(hs) / (float)D + eps);
      for (int d = lane; d < D; d += 64) x[d] *= hinv * ldf(hnw, d);
    }
    wave_lds_sync();
    float ss = 0.f;
    float y[8];   // D <= 512
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const int d = lane + 64 * n;
      float v = 0.f;
      if (d < D) {
        v = x[d];
        if (d < dims && half_layout) {
          const bool first = d < half;
          const int i = first ? d : d - half;
          const float c = cs[i], sn = cs[half + i];
          const float a = x[i], b = x[i + half];
          v = first ? a * c - b * sn : b * c + a * sn;
        } else if (d < dims) {
          const int i = d >> 1;
          const float c = cs[i], sn = cs[half + i];
          const float a = x[d & ~1], b = x[d | 1];
          v = (d & 1) ? b * c + a * sn : a * c - b * sn;
        }
      }
      y[n] = v;
      ss += v * v;
    }
    ss = wave_sum(ss);
    const float inv = unit ? 1.0f / sqrtf(ss / (float)D + eps) : 1.f;
    TA* dst = isq ? row + (size_t)hd * D : (slot >= 0 ? kcache + ((size_t)slot * G + hd) * D : nullptr);
    wave_lds_sync();   // every lane has read its partners before the query row (the source) is overwritten
    if (dst != nullptr) {
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        const int d = lane + 64 * n;
        if (d < D) stf(dst, d, y[n] * inv);
      }
    }
  }
  for (int i = tid; i < G * V; i += blockDim.x) {
    float v = ldf(row + voff, i) + (vb != nullptr ? ldf(vb, i) : 0.f);
    if (vfirst_in != nullptr) v = (1.f - lam) * v + lam * vfirst_in[(size_t)t * G * V + i];
    if (vfirst_out != nullptr) vfirst_out[(size_t)t * G * V + i] = v;
    if (slot >= 0) stf(vcache, (size_t)slot * G * V + i, v);
  }
}

// The same preparation without norms and value mixing, in the half layout, on sizes of whole vectors (D, V, dims / 2 and the
// part offsets multiples of 4): a thread turns four pairs (their partners dims / 2 further on are its own as well), copies
// four unrotated dimensions, or copies four values.  Workgroups (token, slice of the row).
template <typename TA>
__global__ __launch_bounds__(256) void rotate_kv_write_kernel(
    TA* __restrict__ kcache, TA* __restrict__ vcache, TA* __restrict__ qkv, long ld, int koff, int voff,
    const TA* __restrict__ qb, const TA* __restrict__ kb, const TA* __restrict__ vb, const float* __restrict__ cos_sin,
    const int* __restrict__ positions, const int* __restrict__ slot_mapping, int H, int G, int D, int V, int dims) {
  const int t = blockIdx.x;
  const int pos = positions[t];
  if (pos < 0) return;
  const int slot = slot_mapping[t];
  const int half = dims / 2, np = half / 4, per = np + (D - dims) / 4;   // work items of one head
  const int nqk = (H + G) * per, n = nqk + G * V / 4;
  const float* cs = cos_sin + (size_t)pos * dims;
  TA* row = qkv + (size_t)t * ld;
  auto biased = [&](const TA* src, const TA* bias, int i) -> f32x4 {
    f32x4 v = ldf4(src + i);
    if (bias != nullptr) {
      const f32x4 b = ldf4(bias + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += b[e];
    }
    return v;
  };
  for (int it = blockIdx.y * 256 + threadIdx.x; it < n; it += gridDim.y * 256) {
    if (it >= nqk) {
      const int i = 4 * (it - nqk);
      if (slot >= 0) stf4(vcache + (size_t)slot * G * V + i, biased(row + voff, vb, i));
      continue;
    }
    const int hv = it / per, c = it - hv * per;
    const bool isq = hv < H;
    const int at = (isq ? hv : hv - H) * D;
    const TA* src = row + (isq ? 0 : koff);
    const TA* bias = isq ? qb : kb;
    TA* dst = isq ? row : (slot >= 0 ? kcache + (size_t)slot * G * D : nullptr);
    if (dst == nullptr) continue;
    if (c < np) {
      const int i = 4 * c;
      const f32x4 a = biased(src, bias, at + i), b = biased(src, bias, at + half + i);
      const f32x4 co = ldf4(cs + i), sn = ldf4(cs + half + i);
      f32x4 u, w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        u[e] = a[e] * co[e] - b[e] * sn[e];
        w[e] = b[e] * co[e] + a[e] * sn[e];
      }
      stf4(dst + at + i, u);
      stf4(dst + at + half + i, w);
    } else if (!isq || bias != nullptr) {          // unrotated queries without a bias stay as they are
      const int i = dims + 4 * (c - np);
      stf4(dst + at + i, biased(src, bias, at + i));
    }
  }
}

// Entry of pooled block b of a sequence: the block lives with the page that holds its first token.  A page of bs
// tokens holds the first token of at most ppb = ceil(bs / P) blocks.
__device__ __forceinline__ size_t pool_entry(const int* btr, int b, int P, int bs, int ppb) {
  const int page = (int)(((long)b * P) / bs);
  const int first = (int)(((long)page * bs + P - 1) / P);   // the first block that starts in this page
  return (size_t)btr[page] * ppb + (b - first);
}

// Workgroups (token, slice of the row); only tokens that end a block of P work ((pos + 1) % P == 0): the mean, in fp32, of the
// P cached keys and values (as the cache holds them) -> kpool / vpool [pages * ppb][G][D or V] fp32.  Runs after the
// cache write of the same batch, so the block's earlier tokens are in the cache whether this batch or an earlier one
// brought them.
template <typename TA>
__global__ __launch_bounds__(256) void window_pool_kernel(float* __restrict__ kpool, float* __restrict__ vpool,
                                                          const TA* __restrict__ kcache, const TA* __restrict__ vcache,
                                                          const int* __restrict__ block_tables, int max_blocks,
                                                          const int* __restrict__ tok_seq,
                                                          const int* __restrict__ positions, int G, int D, int V, int P,
                                                          int bs, int ppb) {
  const int t = blockIdx.x;
  const int pos = positions[t];
  if (pos < 0 || (pos + 1) % P != 0) return;
  const int b = pos / P;
  const int* btr = block_tables + (size_t)tok_seq[t] * max_blocks;
  const size_t e = pool_entry(btr, b, P, bs, ppb);
  const float invp = 1.0f / (float)P;
  const int GD = G * D, GV = G * V;
  for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < GD + GV; i += gridDim.y * blockDim.x) {
    float a = 0.f;
#pragma unroll 4
    for (int j = b * P; j < b * P + P; ++j) {
      const size_t slot = (size_t)btr[j / bs] * bs + (j % bs);
      a += i < GD ? ldf(kcache, slot * GD + i) : ldf(vcache, slot * GV + (i - GD));
    }
    if (i < GD) kpool[e * GD + i] = a * invp;
    else vpool[e * GV + (i - GD)] = a * invp;
  }
}

// 8 consecutive elements of a cached row as fp32 (one or two 16-byte loads).
__device__ __forceinline__ void load8(const bf16_t* p, float* o) {
  const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = lo_bf(v[i]);
    o[2 * i + 1] = hi_bf(v[i]);
  }
}
__device__ __forceinline__ void load8(const float* p, float* o) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[i] = a[i];
    o[4 + i] = b[i];
  }
}

// One workgroup per (token, key / value head, key split); one wave per query head of the group (further passes when
// the group has more heads than waves).  The visible keys are an ordered list: the nb pooled blocks, then the window's
// tokens.  They come in tiles of KB <= 64 rows staged in LDS as fp32 and shared by the group's heads (the rows' cache
// slots are resolved once per tile; VEC: rows move as 16-byte vectors, D and V multiples of 8); lane l scores row l
// (q . k * scale), the tile joins a running softmax, lane l accumulates value dimensions l, l + 64, ...
// A sink starts the running softmax at (max 0, sum 1).  One split: out[t][head][V] = sum p v / sum, times
// sigmoid(gate) if given.  Several splits (few tokens, many keys: decoding) each take a run of tiles and leave
// (max, sum, unnormalised sum p v) for window_merge_kernel; the sink belongs to split 0.
template <typename TA, int NACC, bool VEC>
__global__ void window_attention_kernel(TA* __restrict__ out, float* __restrict__ pacc, float* __restrict__ pml,
                                        const TA* __restrict__ q, long ldq, const TA* __restrict__ gate, long ldg,
                                        const TA* __restrict__ kcache, const TA* __restrict__ vcache,
                                        const float* __restrict__ kpool, const float* __restrict__ vpool,
                                        const int* __restrict__ block_tables, int max_blocks,
                                        const int* __restrict__ tok_seq, const int* __restrict__ positions, int H, int G,
                                        int D, int V, int window, int P, float scale, int sink, int bs, int ppb, int KB,
                                        int nsplit, int chunk, float softcap, const float* __restrict__ sinkv,
                                        int gate_ph, const float* __restrict__ slopes) {
  extern __shared__ float smem[];
  const int t = blockIdx.x, g = blockIdx.y, split = blockIdx.z;
  const int R = H / G;
  const int p = positions[t];
  if (p < 0) {   // idle row: defined output, nothing read
    if (nsplit == 1)
      for (int i = threadIdx.x; i < R * V; i += blockDim.x) stf(out, (size_t)t * H * V + (size_t)g * R * V + i, 0.f);
    return;
  }
  const int DP = D + 1;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, nw = blockDim.x >> 6;
  float* ktile = smem;                         // [KB][D + 1]
  float* vtile = ktile + (size_t)KB * DP;      // [KB][V]
  float* qs = vtile + (size_t)KB * V;          // [nw][D]
  size_t roff = (size_t)KB * (DP + V) + (size_t)nw * D;
  roff += roff & 1;                            // 8-byte aligned
  long long* rowoff = reinterpret_cast<long long*>(smem + roff);   // [KB] a tile row's cache slot, or -1 - pool entry
  const int lo = chunk > 0 ? p - p % chunk : (window > 0 ? max(0, p - window + 1) : 0);
  const int nb = (window > 0 && P > 0 && p - window + 1 >= P) ? (p - window + 1) / P : 0;
  const int nkeys = nb + (p + 1 - lo);
  const int ntiles = (nkeys + KB - 1) / KB;
  const int tps = (ntiles + nsplit - 1) / nsplit;
  const int tile0 = split * tps, tile1 = min(ntiles, tile0 + tps);
  const int* btr = block_tables + (size_t)tok_seq[t] * max_blocks;
  const int GD = G * D, GV = G * V;
  const bool with_sink = sink && split == 0;
  for (int h0 = 0; h0 < R; h0 += nw) {
    const int hd = g * R + h0 + wave;
    const bool hv = h0 + wave < R;
    float* qq = qs + (size_t)wave * D;
    if (hv)
      for (int d = lane; d < D; d += 64) qq[d] = ldf(q, (size_t)t * ldq + (size_t)hd * D + d);
    const float slope = (slopes != nullptr && hv) ? slopes[hd] : 0.f;
    float m = with_sink ? ((sinkv != nullptr && hv) ? sinkv[hd] : 0.f) : -INFINITY, l = with_sink ? 1.f : 0.f, acc[NACC];
#pragma unroll
    for (int i = 0; i < NACC; ++i) acc[i] = 0.f;
    for (int tile = tile0; tile < tile1; ++tile) {
      const int u0 = tile * KB;
      const int nk = min(KB, nkeys - u0);
      __syncthreads();
      for (int r = tid; r < nk; r += blockDim.x) {
        const int u = u0 + r;
        if (u < nb) {
          rowoff[r] = -1 - (long long)pool_entry(btr, u, P, bs, ppb);
        } else {
          const int j = lo + (u - nb);
          rowoff[r] = (long long)btr[j / bs] * bs + (j % bs);
        }
      }
      __syncthreads();
      if (VEC) {
        const int ckd = D >> 3, cpr = ckd + (V >> 3);
        for (int idx = tid; idx < nk * cpr; idx += blockDim.x) {
          const int r = idx / cpr, c = idx - r * cpr;
          const bool isk = c < ckd;
          const int e8 = 8 * (isk ? c : c - ckd);
          const long long ro = rowoff[r];
          float v8[8];
          if (ro < 0) load8(isk ? kpool + (size_t)(-1 - ro) * GD + (size_t)g * D + e8
                                : vpool + (size_t)(-1 - ro) * GV + (size_t)g * V + e8, v8);
          else load8(isk ? kcache + (size_t)ro * GD + (size_t)g * D + e8 : vcache + (size_t)ro * GV + (size_t)g * V + e8, v8);
          float* dst = isk ? ktile + r * DP + e8 : vtile + r * V + e8;
#pragma unroll
          for (int i = 0; i < 8; ++i) dst[i] = v8[i];
        }
      } else {
        for (int idx = tid; idx < nk * (D + V); idx += blockDim.x) {
          const int r = idx / (D + V), d = idx - r * (D + V);
          const long long ro = rowoff[r];
          float val;
          if (ro < 0) {
            const size_t e = (size_t)(-1 - ro);
            val = d < D ? kpool[e * GD + (size_t)g * D + d] : vpool[e * GV + (size_t)g * V + (d - D)];
          } else {
            val = d < D ? ldf(kcache, (size_t)ro * GD + (size_t)g * D + d)
                        : ldf(vcache, (size_t)ro * GV + (size_t)g * V + (d - D));
          }
          if (d < D) ktile[r * DP + d] = val;
          else vtile[r * V + (d - D)] = val;
        }
      }
      __syncthreads();
      if (hv) {
        float sc = -INFINITY;
        if (lane < nk) {
          const float* kr = ktile + lane * DP;
          float a = 0.f;
          for (int d = 0; d < D; ++d) a = fmaf(qq[d], kr[d], a);
          sc = a * scale;
          if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
          if (slopes != nullptr) sc -= slope * (float)(p - (lo + u0 + lane - nb));
        }
        const float mn = fmaxf(m, wave_max(sc));
        const float alpha = m == -INFINITY ? 0.f : expf(m - mn);
        const float pj = lane < nk ? expf(sc - mn) : 0.f;
        l = l * alpha + wave_sum(pj);
        m = mn;
#pragma unroll
        for (int i = 0; i < NACC; ++i) acc[i] *= alpha;
        for (int jj = 0; jj < nk; ++jj) {
          const float pb = __shfl(pj, jj, WAVE);
#pragma unroll
          for (int i = 0; i < NACC; ++i) {
            const int d = lane + 64 * i;
            if (d < V) acc[i] = fmaf(pb, vtile[jj * V + d], acc[i]);
          }
        }
      }
    }
    if (hv && nsplit == 1) {
#pragma unroll
      for (int i = 0; i < NACC; ++i) {
        const int d = lane + 64 * i;
        if (d < V) {
          float o = acc[i] / l;
          if (gate != nullptr)
            o *= 1.f / (1.f + expf(-ldf(gate, (size_t)t * ldg + (gate_ph ? (size_t)hd : (size_t)hd * V + d))));
          stf(out, (size_t)t * H * V + (size_t)hd * V + d, o);
        }
      }
    } else if (hv) {
      const size_t rec = ((size_t)t * H + hd) * nsplit + split;
#pragma unroll
      for (int i = 0; i < NACC; ++i) {
        const int d = lane + 64 * i;
        if (d < V) pacc[rec * V + d] = acc[i];
      }
      if (lane == 0) {
        pml[rec * 2] = m;           // -inf and 0 for a split without tiles and without the sink
        pml[rec * 2 + 1] = l;
      }
    }
  }
}

// out[t][head] = sum_s e^(m_s - M) acc_s / sum_s e^(m_s - M) l_s over the key splits (at most 64), times sigmoid(gate) if
// given.  One wave per (token, head): lane s weighs split s, then every lane sums its value dimensions, 8 splits' loads in
// flight (a load under the weight's branch waited for each split: 97 tokens, 16 heads of 128, 6 splits 7.4 -> 4.3 us).
template <typename TA>
__global__ __launch_bounds__(64) void window_merge_kernel(TA* __restrict__ out, const float* __restrict__ pacc,
                                                          const float* __restrict__ pml, const TA* __restrict__ gate,
                                                          long ldg, const int* __restrict__ positions, int H, int V,
                                                          int nsplit, int gate_ph) {
  const int t = blockIdx.x, hd = blockIdx.y, lane = threadIdx.x;
  if (positions[t] < 0) {
    for (int d = lane; d < V; d += 64) stf(out, (size_t)t * H * V + (size_t)hd * V + d, 0.f);
    return;
  }
  const size_t rec0 = ((size_t)t * H + hd) * nsplit;
  float ms = -INFINITY, ls = 0.f;
  if (lane < nsplit) {
    ms = pml[(rec0 + lane) * 2];
    ls = pml[(rec0 + lane) * 2 + 1];
  }
  const float M = wave_max(ms);
  float wt = ms == -INFINITY ? 0.f : expf(ms - M);
  wt /= wave_sum(wt * ls);
  for (int d0 = 0; d0 < V; d0 += 64) {            // every lane stays in the loop: the shuffles read all of them
    const int d = d0 + lane, dc = min(d, V - 1);
    float a = 0.f;
    for (int s0 = 0; s0 < nsplit; s0 += 8) {      // 8 splits' loads in flight, at clamped places
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = pacc[(rec0 + min(s0 + u, nsplit - 1)) * V + dc];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float w = __shfl(wt, s0 + u, WAVE);       // (0 past the last split, and for a split without keys, which left nothing)
        a = w != 0.f ? fmaf(w, x[u], a) : a;
      }
    }
    if (d >= V) continue;
    if (gate != nullptr)
      a *= 1.f / (1.f + expf(-ldf(gate, (size_t)t * ldg + (gate_ph ? (size_t)hd : (size_t)hd * V + d))));
    stf(out, (size_t)t * H * V + (size_t)hd * V + d, a);
  }
}

// The same attention on the matrix cores for prompts in bf16 (D % 8 == 0, V % 16 == 0, R = H / G a power of two <= 16).
// A workgroup of 4 waves takes TPB consecutive tokens of one sequence and one key / value head; a wave owns NCB blocks
// of 16 query columns, a column being one (token, query head of the group) pair, 16 / R tokens per block.  The keys of
// the workgroup are the ordered list [pooled blocks 0 .. nb(last token) | tokens lo(first token) .. last token]; 32 of
// them per step are staged in LDS as bf16 (pooled rows converted from fp32) and shared by the waves, each column masks
// what its own token does not see:
//   S^T[key][column] = K Q^T      A = 16 staged key rows, B = the columns' queries (registers)
//   O[column][d]    += P V        A = the 32 keys' probabilities (registers, keys in the order the S^T tiles left
//                                 them), B = the staged value columns through the transposing LDS read
// scores, softmax and sums in fp32, the weights applied as two bf16 terms; a sink starts every column at (max 0, sum 1).
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

template <int NKK, int NVB, int NCB, bool PF>
__global__ __launch_bounds__(256) void window_attention_mfma_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, long ldq, const bf16_t* __restrict__ gate, long ldg,
    const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache, const float* __restrict__ kpool,
    const float* __restrict__ vpool, const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ cu_q,
    const int* __restrict__ positions, int H, int G, int D, int V, int window, int P, float scale, int sink, int bs,
    int ppb, int R, int chunk, float softcap, const float* __restrict__ sinkv, int gate_ph,
    const float* __restrict__ slopes) {
  extern __shared__ __attribute__((aligned(16))) char smem_w[];
  const int seq = blockIdx.z, g = blockIdx.y;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g4 = lane >> 4;
  const int TPC = 16 / R, TPB = 4 * NCB * TPC;
  const int tq0 = cu_q[seq] + blockIdx.x * TPB, tend = cu_q[seq + 1];
  if (tq0 >= tend) return;
  const int p_first = positions[tq0];
  const int nval = min(TPB, tend - tq0);
  if (p_first < 0) {   // idle rows: defined output
    for (int i = tid; i < nval * R * V; i += 256) {
      const int tt = i / (R * V), r = i - tt * (R * V);
      out[(size_t)(tq0 + tt) * H * V + (size_t)g * R * V + r] = 0;
    }
    return;
  }
  const int p_last = p_first + nval - 1;
  const int rowk = (D + 8) * 2, rowv = (V + 8) * 2;      // LDS row bytes
  char* klds = smem_w;                                   // [32][D + 8] bf16
  char* vlds = smem_w + 32 * rowk;                       // [32][V + 8] bf16
  const bool win = window > 0;
  // the first position a token at p sees: its chunk's first, the window's first, or 0 (never decreasing in p)
  auto lo_of = [&](int p) { return chunk > 0 ? p - p % chunk : (win ? max(0, p - window + 1) : 0); };
  const int lo_min = lo_of(p_first);
  const int nb_max = (win && P > 0 && p_last - window + 1 >= P) ? (p_last - window + 1) / P : 0;
  const int nkeys = nb_max + (p_last + 1 - lo_min);
  const int nsteps = (nkeys + 31) / 32;
  const int* btr = block_tables + (size_t)seq * max_blocks;
  const int GD = G * D, GV = G * V;
  const int ckd = D / 8, ckv = V / 8, cpr = ckd + ckv;   // 16-byte chunks per staged row
  const int nkk = (D + 31) / 32, nvb = V / 16;
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  // this lane's column in every block of the wave: token, position, first visible token, visible pooled blocks
  int c_tok[NCB], c_p[NCB], c_lo[NCB], c_nb[NCB];
  bf16x8 qf[NCB][NKK];
  int w_pmin = 0x7fffffff, w_pmax = -1;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const int toff = (wave * NCB + cb) * TPC + li / R;
    const bool ok = toff < nval;
    c_tok[cb] = tq0 + toff;
    c_p[cb] = ok ? p_first + toff : -1;
    c_lo[cb] = ok ? lo_of(c_p[cb]) : 0;
    c_nb[cb] = (ok && win && P > 0 && c_p[cb] - window + 1 >= P) ? (c_p[cb] - window + 1) / P : 0;
    const int hd = g * R + li % R;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      const int piece = 32 * kk + 8 * g4;
      u32x4 v = zero;
      if (ok && piece < D) v = *reinterpret_cast<const u32x4*>(q + (size_t)c_tok[cb] * ldq + (size_t)hd * D + piece);
      qf[cb][kk] = __builtin_bit_cast(bf16x8, v);
    }
    const int t_lo = (wave * NCB + cb) * TPC, t_hi = min(t_lo + TPC, nval) - 1;
    if (t_lo < nval) {
      w_pmin = min(w_pmin, p_first + t_lo);
      w_pmax = max(w_pmax, p_first + t_hi);
    }
  }
  const bool w_any = w_pmax >= 0;
  const int w_lo = w_any ? lo_of(w_pmin) : 0;
  const int w_nb = (w_any && win && P > 0 && w_pmax - window + 1 >= P) ? (w_pmax - window + 1) / P : 0;
  f32x4 o[NCB][NVB];
  float m_run[NCB], l_run[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    m_run[cb] = sink ? (sinkv != nullptr ? sinkv[g * R + li % R] : 0.f) : -INFINITY;
    l_run[cb] = sink ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NVB; ++n) o[cb][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float slope = slopes != nullptr ? slopes[g * R + li % R] : 0.f;   // the head of this lane's columns
  const int qd = li >> 2, pd = li & 3;
  // Staging: every thread moves NST 16-byte chunks of a step's 32 rows.  PF: the chunks of step s + 1 are loaded into
  // registers before step s is computed and written to LDS after it, so the cache reads run under the MFMAs -- for
  // grids of at most one workgroup per CU, where nothing else hides them; larger grids run the variant without the
  // held registers, at twice the waves per SIMD.
  constexpr int NST = (NKK * 4 + NVB * 2 + 7) / 8;
  u32x4 pre[NST];
  auto stage_load = [&](int u0) {
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int idx = tid + 256 * i;
      u32x4 v = zero;
      if (idx < 32 * cpr) {
        const int r = idx / cpr, c = idx - r * cpr, u = u0 + r;
        const bool isk = c < ckd;
        const int e8 = 8 * (isk ? c : c - ckd);
        if (u < nb_max) {
          const size_t e = pool_entry(btr, u, P, bs, ppb);
          const float* src = isk ? kpool + e * GD + (size_t)g * D + e8 : vpool + e * GV + (size_t)g * V + e8;
          const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
          v = u32x4{pack_bf2(a[0], a[1]), pack_bf2(a[2], a[3]), pack_bf2(b[0], b[1]), pack_bf2(b[2], b[3])};
        } else if (u < nkeys) {
          const int j = lo_min + (u - nb_max);
          const size_t slot = (size_t)btr[j / bs] * bs + (j % bs);
          v = isk ? *reinterpret_cast<const u32x4*>(kcache + slot * GD + (size_t)g * D + e8)
                  : *reinterpret_cast<const u32x4*>(vcache + slot * GV + (size_t)g * V + e8);
        }
      }
      pre[i] = v;
    }
  };
  auto stage_store = [&]() {
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int idx = tid + 256 * i;
      if (idx < 32 * cpr) {
        const int r = idx / cpr, c = idx - r * cpr;
        const bool isk = c < ckd;
        const int e8 = 8 * (isk ? c : c - ckd);
        *reinterpret_cast<u32x4*>((isk ? klds + r * rowk : vlds + r * rowv) + 2 * e8) = pre[i];
      }
    }
  };
  if (PF) stage_load(0);
  for (int step = 0; step < nsteps; ++step) {
    const int u0 = step * 32;
    __syncthreads();          // the previous step's fragments have been read
    if (PF) {
      stage_store();
    } else {                  // chunk by chunk: no registers held across the step
      for (int idx = tid; idx < 32 * cpr; idx += 256) {
        const int r = idx / cpr, c = idx - r * cpr, u = u0 + r;
        const bool isk = c < ckd;
        const int e8 = 8 * (isk ? c : c - ckd);
        u32x4 v = zero;
        if (u < nb_max) {
          const size_t e = pool_entry(btr, u, P, bs, ppb);
          const float* src = isk ? kpool + e * GD + (size_t)g * D + e8 : vpool + e * GV + (size_t)g * V + e8;
          const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
          v = u32x4{pack_bf2(a[0], a[1]), pack_bf2(a[2], a[3]), pack_bf2(b[0], b[1]), pack_bf2(b[2], b[3])};
        } else if (u < nkeys) {
          const int j = lo_min + (u - nb_max);
          const size_t slot = (size_t)btr[j / bs] * bs + (j % bs);
          v = isk ? *reinterpret_cast<const u32x4*>(kcache + slot * GD + (size_t)g * D + e8)
                  : *reinterpret_cast<const u32x4*>(vcache + slot * GV + (size_t)g * V + e8);
        }
        *reinterpret_cast<u32x4*>((isk ? klds + r * rowk : vlds + r * rowv) + 2 * e8) = v;
      }
    }
    __syncthreads();
    if (PF && step + 1 < nsteps) stage_load(u0 + 32);
    // keys of this step that any column of the wave can see: pooled blocks below w_nb, tokens w_lo .. w_pmax
    bool any = false;
    if (w_any) {
      if (u0 < nb_max) any = u0 < w_nb;
      const int j_first = lo_min + max(u0 - nb_max, 0), j_last = lo_min + (u0 + 31 - nb_max);
      if (u0 + 31 >= nb_max && j_first <= w_pmax && j_last >= w_lo) any = true;
    }
    if (!any) continue;
    // every staged key fragment is read once and serves all column blocks of the wave
    f32x4 sacc[NCB][2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) sacc[cb][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        if (kk < nkk) {
          const int piece = 32 * kk + 8 * g4;
          bf16x8 ka = __builtin_bit_cast(bf16x8, zero);
          if (piece < D) ka = *reinterpret_cast<const bf16x8*>(klds + (16 * m + li) * rowk + 2 * piece);
#pragma unroll
          for (int cb = 0; cb < NCB; ++cb)
            sacc[cb][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[cb][kk], sacc[cb][m], 0, 0, 0);
        }
      }
    }   // sacc[cb][m][i] = S[key u0 + 16 m + 4 g4 + i][column li of block cb]
    bf16x8 pa[NCB], pl[NCB];   // slot j < 4: key 4 g4 + j; slot j >= 4: key 16 + 4 g4 + (j - 4)
    float a_i[NCB][4];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      float tmax = -INFINITY;
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int u = u0 + 16 * m + 4 * g4 + i;
          bool vis;
          if (u < nb_max) vis = u < c_nb[cb];
          else {
            const int j = lo_min + (u - nb_max);
            vis = j <= c_p[cb] && j >= c_lo[cb];
          }
          float v = -INFINITY;
          if (vis) {
            v = sacc[cb][m][i] * scale;
            if (softcap > 0.f) v = softcap * tanhf(v / softcap);
            if (slopes != nullptr) v -= slope * (float)(c_p[cb] - (lo_min + (u - nb_max)));
          }
          sacc[cb][m][i] = v;
          tmax = fmaxf(tmax, v);
        }
      tmax = lane_max<16>(tmax);
      tmax = lane_max<32>(tmax);
      const float m_new = fmaxf(m_run[cb], tmax);
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;      // a column that has seen nothing yet
      const float alpha = m_run[cb] == -INFINITY ? 0.f : expf(m_run[cb] - m_ref);
      float rsum = 0.f;
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pv = expf(sacc[cb][m][i] - m_ref);
          sacc[cb][m][i] = pv;
          rsum += pv;
        }
      rsum = lane_sum<16>(rsum);
      rsum = lane_sum<32>(rsum);
      l_run[cb] = l_run[cb] * alpha + rsum;
      m_run[cb] = m_new;
#pragma unroll
      for (int i = 0; i < 4; ++i) a_i[cb][i] = __shfl(alpha, g4 * 4 + i, WAVE);
      // the fp32 weights enter the product as two bf16 terms (p = hi + lo, |lo| <= 2^-9 p): 16 bits of each weight
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        pa[cb][j] = (__bf16)sacc[cb][0][j];
        pa[cb][4 + j] = (__bf16)sacc[cb][1][j];
        pl[cb][j] = (__bf16)(sacc[cb][0][j] - (float)pa[cb][j]);
        pl[cb][4 + j] = (__bf16)(sacc[cb][1][j] - (float)pa[cb][4 + j]);
      }
    }
    const int r0 = 4 * g4 + qd, r1 = r0 + 16;
#pragma unroll
    for (int n = 0; n < NVB; ++n) {
      if (n < nvb) {
        const int col = 16 * n + 4 * pd;
        const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vlds + r0 * rowv + 2 * col));
        const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vlds + r1 * rowv + 2 * col));
        bf16x8 vb;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vb[j] = v0[j]; vb[4 + j] = v1[j]; }
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
#pragma unroll
          for (int i = 0; i < 4; ++i) o[cb][n][i] *= a_i[cb][i];
          o[cb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[cb], vb, o[cb][n], 0, 0, 0);
          o[cb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[cb], vb, o[cb][n], 0, 0, 0);
        }
      }
    }
  }
  // o[cb][n][i] = O[column 4 g4 + i][d 16 n + li]; a column's sum lives in the lanes with li == column
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    float l_i[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) l_i[i] = __shfl(l_run[cb], g4 * 4 + i, WAVE);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 4 * g4 + i;
      const int toff = (wave * NCB + cb) * TPC + c / R;
      if (toff >= nval) continue;
      const int t = tq0 + toff, hd = g * R + c % R;
      const float inv = 1.f / l_i[i];
#pragma unroll
      for (int n = 0; n < NVB; ++n)
        if (n < nvb) {
          const int d = 16 * n + li;
          float y = o[cb][n][i] * inv;
          if (gate != nullptr)
            y *= 1.f / (1.f + expf(-bf2f(gate[(size_t)t * ldg + (gate_ph ? (size_t)hd : (size_t)hd * V + d)])));
          out[(size_t)t * H * V + (size_t)hd * V + d] = f2bf(y);
        }
    }
  }
}

// The prompt kernel without pooled blocks, for exact sizes (DK key, DV value dimensions) and pages of a power of two.  The
// orientation of the products is the one above; what differs:
//   * 8 waves in two groups: both groups own the same tokens (a wave one block of 16 columns), group k takes the keys
//     [32 k, 32 k + 32) of every 64-key step with a running softmax of its own, and the two are merged at the end;
//   * one column block a wave is at most 128 registers, so two workgroups share a CU: a step is a chain of LDS reads, shuffles
//     and about 350 vector instructions a block (2 us for a lone workgroup), and four waves per SIMD hide each other's.
//     With two blocks a wave (210 registers, one workgroup on a CU, each staged key used twice) a step is no shorter and the
//     longest sequence of a batch decides: 16 query heads over 4 of 128, five prompts of 153 - 459 tokens and three single
//     tokens behind 640 - 700 39.6 -> 27.8 us, 512 fresh tokens 23.9 -> 22.0, 1024 38.6 -> 32.1, 97 behind 1000 23.4 ->
//     20.6 (17.3 with the merge as it is now), 2048 47.4 -> 47.2 (with the merge where there is one);
//   * two LDS buffers, one barrier per step: while a step is computed the next one is stored and the one after next is
//     loaded into registers, its page numbers a step earlier still; a thread always moves one row's pieces;
//   * scores in base 2 (scale and slopes carry log2 e), no mask arithmetic on slices that every column of the wave sees,
//     accumulators rescaled only when some column's maximum moved, sums kept per lane until the end;
//   * where the tiles are few (a short portion behind a long cached one), nsplit workgroups share a tile's steps and leave
//     (max, sum, unnormalised sum) for window_merge_kernel: 97 tokens behind 1000 32.7 us in one piece, 17.3 us in 6 with the
//     merge.  (A template flag: the arithmetic of the splits costs the whole walk 8%.)
template <int DK, int DV, bool SPLIT>
__global__ __launch_bounds__(512, 4) void window_prompt_kernel(
    bf16_t* __restrict__ out, float* __restrict__ pacc, float* __restrict__ pml, const bf16_t* __restrict__ q, long ldq,
    const bf16_t* __restrict__ gate, long ldg, const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ cu_q, const int* __restrict__ positions,
    int H, int G, int window, float scale, int sink, int bshift, int nsplit, int R, int chunk, float softcap,
    const float* __restrict__ sinkv, int gate_ph, const float* __restrict__ slopes) {
  constexpr int NCB = 1, NKK = DK / 32, NVB = DV / 16, KT = 64;      // NCB: column blocks of a wave
  constexpr int ROWK = (DK + 8) * 2, ROWV = (DV + 8) * 2, BUF = KT * (ROWK + ROWV);   // LDS bytes
  constexpr int CK = DK / 8, CV = DV / 8, NST = (CK + CV + 7) / 8;                   // 16-byte pieces; per thread
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(16))) char smem_p[];
  const int seq = blockIdx.z, g = blockIdx.y;
  const int tid = threadIdx.x, wave = (tid >> 6) & 3, grp = tid >> 8, lane = tid & 63, li = lane & 15, g4 = lane >> 4;
  const int TPC = 16 / R, TPB = 4 * NCB * TPC;
  const int split = SPLIT ? blockIdx.x % nsplit : 0;
  const int tq0 = cu_q[seq] + (SPLIT ? blockIdx.x / nsplit : blockIdx.x) * TPB, tend = cu_q[seq + 1];
  if (tq0 >= tend) return;
  const int p_first = positions[tq0];
  const int nval = min(TPB, tend - tq0);
  if (p_first < 0) {   // idle rows: defined output
    if (SPLIT) return;          // (the merge's business)
    for (int i = tid; i < nval * R * DV; i += 512) {
      const int tt = i / (R * DV), r = i - tt * (R * DV);
      out[(size_t)(tq0 + tt) * H * DV + (size_t)g * R * DV + r] = 0;
    }
    return;
  }
  const int p_last = p_first + nval - 1;
  auto lo_of = [&](int p) { return chunk > 0 ? p - p % chunk : (window > 0 ? max(0, p - window + 1) : 0); };
  const int lo_min = lo_of(p_first);
  const int nkeys = p_last + 1 - lo_min;
  const int ntot = (nkeys + KT - 1) / KT, per = SPLIT ? max(2, (ntot + nsplit - 1) / nsplit) : ntot;
  const int step0 = split * per, nsteps = min(ntot, step0 + per);      // this split's steps
  if (SPLIT && step0 >= ntot) {   // none (split 0 always has one)
    for (int i = tid; i < nval * R; i += 512) {
      const int tt = i / R;
      const size_t rec = ((size_t)(tq0 + tt) * H + g * R + (i - tt * R)) * nsplit + split;
      pml[rec * 2] = -INFINITY;
      pml[rec * 2 + 1] = 0.f;
    }
    return;
  }
  const int* btr = block_tables + (size_t)seq * max_blocks;
  const int GD = G * DK, GV = G * DV, bmask = (1 << bshift) - 1;
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  int c_tok[NCB], c_p[NCB], c_lo[NCB];
  bf16x8 qf[NCB][NKK];
  const int hd = g * R + li % R;                 // the head of this lane's columns
  int w_pmin = 0x7fffffff, w_pmax = -1;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const int toff = (wave * NCB + cb) * TPC + li / R;
    const bool ok = toff < nval;
    c_tok[cb] = tq0 + toff;
    c_p[cb] = ok ? p_first + toff : -1;
    c_lo[cb] = ok ? lo_of(c_p[cb]) : 0;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      u32x4 v = zero;
      if (ok) v = *reinterpret_cast<const u32x4*>(q + (size_t)c_tok[cb] * ldq + (size_t)hd * DK + 32 * kk + 8 * g4);
      qf[cb][kk] = __builtin_bit_cast(bf16x8, v);
    }
    const int t_lo = (wave * NCB + cb) * TPC, t_hi = min(t_lo + TPC, nval) - 1;
    if (t_lo < nval) {
      w_pmin = min(w_pmin, p_first + t_lo);
      w_pmax = max(w_pmax, p_first + t_hi);
    }
  }
  const bool w_any = w_pmax >= 0;
  const int w_lo = w_any ? lo_of(w_pmin) : 0, w_hi_lo = w_any ? lo_of(w_pmax) : 0;   // first key any / every column sees
  const bool with_sink = sink && grp == 0 && split == 0;
  const float sc2 = scale * LOG2E;
  const float slope2 = slopes != nullptr ? slopes[hd] * LOG2E : 0.f;
  f32x4 o[NCB][NVB];
  float m_run[NCB], l_run[NCB];                  // l_run: this lane's keys only
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    m_run[cb] = with_sink ? (sinkv != nullptr ? sinkv[hd] * LOG2E : 0.f) : -INFINITY;
    l_run[cb] = with_sink && g4 == 0 ? 1.f : 0.f;
#pragma unroll
    for (int n = 0; n < NVB; ++n) o[cb][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int qd = li >> 2, pd = li & 3;
  // staging: thread -> row tid / 8 of the step, pieces tid % 8 + 8 i of [K row | V row]
  const int sr = tid >> 3, sc = tid & 7;
  u32x4 pre[NST];
  auto page_of = [&](int step) -> int {
    const int u = step * KT + sr;
    return u < nkeys ? btr[(lo_min + u) >> bshift] : -1;
  };
  auto stage_load = [&](int step, int page) {
    const size_t slot = page >= 0 ? ((size_t)page << bshift) + ((lo_min + step * KT + sr) & bmask) : 0;
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = sc + 8 * i;
      u32x4 v = zero;
      if (page >= 0 && c < CK + CV)
        v = c < CK ? *reinterpret_cast<const u32x4*>(kcache + slot * GD + (size_t)g * DK + 8 * c)
                   : *reinterpret_cast<const u32x4*>(vcache + slot * GV + (size_t)g * DV + 8 * (c - CK));
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
  stage_load(step0, page_of(step0));
  stage_store(smem_p + (step0 & 1) * BUF);
  int page = step0 + 1 < nsteps ? page_of(step0 + 1) : -1;
  if (step0 + 1 < nsteps) stage_load(step0 + 1, page);
  page = step0 + 2 < nsteps ? page_of(step0 + 2) : -1;
  __syncthreads();
  for (int step = step0; step < nsteps; ++step) {
    char* buf = smem_p + (step & 1) * BUF;
    if (step + 1 < nsteps) {
      stage_store(smem_p + ((step + 1) & 1) * BUF);
      if (step + 2 < nsteps) {
        stage_load(step + 2, page);
        page = step + 3 < nsteps ? page_of(step + 3) : -1;
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
      bf16x8 pa[NCB], pl[NCB];   // slot j < 4: key 4 g4 + j; slot j >= 4: key 16 + 4 g4 + (j - 4)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        if (softcap > 0.f) {
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) sacc[cb][m][i] = softcap * LOG2E * tanhf(sacc[cb][m][i] * scale / softcap);
        } else {
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) sacc[cb][m][i] *= sc2;
        }
        if (slopes != nullptr) {
          const float d0 = (float)(c_p[cb] - j0 - 4 * g4);
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) sacc[cb][m][i] = fmaf(-slope2, d0 - (float)(16 * m + i), sacc[cb][m][i]);
        }
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
        // the fp32 weights enter the product as two bf16 terms (p = hi + lo, |lo| <= 2^-9 p): 16 bits of each weight
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pa[cb][j] = (__bf16)sacc[cb][0][j];
          pa[cb][4 + j] = (__bf16)sacc[cb][1][j];
          pl[cb][j] = (__bf16)(sacc[cb][0][j] - (float)pa[cb][j]);
          pl[cb][4 + j] = (__bf16)(sacc[cb][1][j] - (float)pa[cb][4 + j]);
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
        for (int cb = 0; cb < NCB; ++cb) {
          o[cb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[cb], vb, o[cb][n], 0, 0, 0);
          o[cb][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[cb], vb, o[cb][n], 0, 0, 0);
        }
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
    const float lsum = l_run[cb] * f0 + b[(4 * NVB + 1) * 64] * f1, inv = SPLIT ? 1.f : 1.f / lsum;
    const float m2 = M * 0.6931471805599453f;       // -inf and sum 0: no key of this split is seen
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 4 * g4 + i;
      const float w0 = __shfl(f0 * inv, c, WAVE), w1 = __shfl(f1 * inv, c, WAVE);
      const float mt = SPLIT ? __shfl(m2, c, WAVE) : 0.f, lt = SPLIT ? __shfl(lsum, c, WAVE) : 0.f;
      const int toff = (wave * NCB + cb) * TPC + c / R;
      if (toff >= nval) continue;
      const int t = tq0 + toff, h = g * R + c % R;
      if constexpr (SPLIT) {
        const size_t rec = ((size_t)t * H + h) * nsplit + split;
#pragma unroll
        for (int n = 0; n < NVB; ++n) pacc[rec * DV + 16 * n + li] = o[cb][n][i] * w0 + b[(4 * n + i) * 64] * w1;
        if (li == 0) {
          pml[rec * 2] = mt;
          pml[rec * 2 + 1] = lt;
        }
        continue;
      }
      float s = 1.f;
      if (gate != nullptr && gate_ph) s = 1.f / (1.f + expf(-bf2f(gate[(size_t)t * ldg + h])));
#pragma unroll
      for (int n = 0; n < NVB; ++n) {
        const int d = 16 * n + li;
        float y = o[cb][n][i] * w0 + b[(4 * n + i) * 64] * w1;
        if (gate != nullptr && !gate_ph) s = 1.f / (1.f + expf(-bf2f(gate[(size_t)t * ldg + (size_t)h * DV + d])));
        out[(size_t)t * H * DV + (size_t)h * DV + d] = f2bf(y * s);
      }
    }
  }
}

// Single tokens on the matrix cores (no pooled blocks, DK key and value dimensions, pages of a power of two, at most 16 query
// heads per key head): workgroups (token, key head, key split) of NW waves.  A wave walks its own 32-key tiles without a
// workgroup barrier: keys go from the cache straight into MFMA operands (a lane loads 8 dimensions of one key), values
// through the wave's LDS rows for the transposing read; the 16 columns of the products are the group's heads (padded).  The
// waves merge in LDS; one split writes the result, several leave (max, sum, unnormalised sum) for window_merge_kernel.
// AHEAD: a tile's loads go out ahead of the softmax and the second product of the one before, at a sixth more registers; for few tokens,
// whose workgroups have a CU each (16 heads over 4 of 128, 32 tokens behind up to 545 keys 15.7 -> 14.1 us, 1500 26.0 -> 24.9, 4 in splits
// 10.2 -> 9.7; 32 over 8, 16 tokens 15.3 -> 13.6; 32 behind 1500 30.7 / 32.3 with it, 31.4 without).  Keys past the last repeat it, where skipping
// them took a branch a load.
// A tile is a chain of loads and LDS of 2.5 us, the merge's launch 4 us: 8 waves take the tiles of 512 keys in two rounds and
// need no splits.  16 heads over 4 of 128, us, 4 waves with splits and their merge -> 8 waves: 32 tokens behind up to 545 keys
// 17.5 -> 13.9, behind 100 10.0 -> 6.2, 64 behind 545 20.4 -> 14.8; with half the splits one token behind 1024 14.6 -> 12.5, 8
// behind 1500 without a window 21.3 -> 15.3.  16 waves (no splits at all) do not fit 128 registers at 128 dimensions: 19.1.
template <int DK, int NW, bool AHEAD>
__global__ __launch_bounds__(64 * NW) void window_token_kernel(
    bf16_t* __restrict__ out, float* __restrict__ pacc, float* __restrict__ pml, const bf16_t* __restrict__ q, long ldq,
    const bf16_t* __restrict__ gate, long ldg, const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ tok_seq,
    const int* __restrict__ positions, int H, int G, int window, float scale, int sink, int bshift, int nsplit, int chunk,
    float softcap, const float* __restrict__ sinkv, int gate_ph, const float* __restrict__ slopes) {
  constexpr int NKK = DK / 32, NVB = DK / 16, C8 = DK / 8, ROWV = (DK + 8) * 2, NV = 32 * C8 / 64;
  constexpr float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;
  __shared__ __attribute__((aligned(16))) char vrows[NW][32 * ROWV];   // a wave's values; later its sums [R][DK] fp32
  __shared__ float ml[NW][16][2];
  const int t = blockIdx.x, g = blockIdx.y, split = blockIdx.z, R = H / G;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g4 = lane >> 4;
  const int p = positions[t];
  if (p < 0) {   // idle row: defined output, nothing read
    if (nsplit == 1)
      for (int i = tid; i < R * DK; i += 64 * NW) out[(size_t)t * H * DK + (size_t)g * R * DK + i] = 0;
    return;
  }
  const int lo = chunk > 0 ? p - p % chunk : (window > 0 ? max(0, p - window + 1) : 0);
  const int ntiles = (p + 1 - lo + 31) / 32, tps = (ntiles + nsplit - 1) / nsplit;
  const int tile0 = split * tps, tile1 = min(ntiles, tile0 + tps);
  const int* btr = block_tables + (size_t)tok_seq[t] * max_blocks;
  const int GD = G * DK, bmask = (1 << bshift) - 1;
  const int hd = g * R + (li < R ? li : 0);       // padding columns repeat the first head
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  bf16x8 qf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)
    qf[kk] = *reinterpret_cast<const bf16x8*>(q + (size_t)t * ldq + (size_t)hd * DK + 32 * kk + 8 * g4);
  const float sc2 = scale * LOG2E, slope2 = slopes != nullptr ? slopes[hd] * LOG2E : 0.f;
  const bool with_sink = sink && split == 0 && wave == 0;
  float m_run = with_sink ? (sinkv != nullptr ? sinkv[hd] * LOG2E : 0.f) : -INFINITY;
  float l_run = with_sink && g4 == 0 ? 1.f : 0.f;
  f32x4 o[NVB];
#pragma unroll
  for (int n = 0; n < NVB; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  char* vl = vrows[wave];
  const int qd = li >> 2, pd = li & 3;
  // keys past the last (the tile's rest) repeat it: their scores are masked, their values zeroed on the way to LDS
  int slot[2];                                    // cache slots of keys 16 m + li of the tile that is loaded next
  bf16x8 kf[2][NKK];
  u32x4 vv[NV];
  auto slots_of = [&](int tile) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int j = min(lo + tile * 32 + 16 * m + li, p);
      slot[m] = (btr[j >> bshift] << bshift) + (j & bmask);
    }
  };
  auto load_k = [&]() {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk)
        kf[m][kk] = *reinterpret_cast<const bf16x8*>(kcache + (size_t)slot[m] * GD + (size_t)g * DK + 32 * kk + 8 * g4);
  };
  auto load_v = [&]() {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = lane + 64 * i, r = idx / C8, c = idx - r * C8;
      const int s0 = __shfl(slot[0], r & 15, WAVE), s1 = __shfl(slot[1], r & 15, WAVE), sv = r < 16 ? s0 : s1;
      vv[i] = *reinterpret_cast<const u32x4*>(vcache + (size_t)sv * GD + (size_t)g * DK + 8 * c);
    }
  };
  if (AHEAD && tile0 + wave < tile1) {
    slots_of(tile0 + wave);
    load_k();
    load_v();
    slots_of(tile0 + wave + NW);
  }
  for (int tile = tile0 + wave; tile < tile1; tile += NW) {
    const int j0 = lo + tile * 32;
    if constexpr (!AHEAD) {
      slots_of(tile);
      load_k();
      load_v();
    }
    f32x4 sacc[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      sacc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) sacc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[m][kk], qf[kk], sacc[m], 0, 0, 0);
    }   // sacc[m][i] = S[key j0 + 16 m + 4 g4 + i][head column li]
    wave_lds_sync();                              // the previous tile's values have been read
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = lane + 64 * i, r = idx / C8, c = idx - r * C8;
      *reinterpret_cast<u32x4*>(vl + r * ROWV + 16 * c) = j0 + r <= p ? vv[i] : zero;
    }
    if (AHEAD && tile + NW < tile1) {             // the next tile is under way while this one is weighed and summed
      load_k();
      load_v();
      slots_of(tile + 2 * NW);
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + 16 * m + 4 * g4 + i;
        float v = softcap > 0.f ? softcap * LOG2E * tanhf(sacc[m][i] * scale / softcap) : sacc[m][i] * sc2;
        v = j <= p ? fmaf(-slope2, (float)(p - j), v) : -INFINITY;
        sacc[m][i] = v;
        tmax = fmaxf(tmax, v);
      }
    tmax = lane_max<16>(tmax);
    tmax = lane_max<32>(tmax);
    const float m_new = fmaxf(m_run, tmax);       // finite: the tile's first key is seen
    const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
    bf16x8 pa, pl;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w = __builtin_amdgcn_exp2f(sacc[m][i] - m_new);
        l_run += w;
        pa[4 * m + i] = (__bf16)w;
        pl[4 * m + i] = (__bf16)(w - (float)pa[4 * m + i]);
      }
    float a_i[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a_i[i] = __shfl(alpha, g4 * 4 + i, WAVE);
    wave_lds_sync();
    const int r0 = 4 * g4 + qd, r1 = r0 + 16;
#pragma unroll
    for (int n = 0; n < NVB; ++n) {
      const int col = 16 * n + 4 * pd;
      const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vl + r0 * ROWV + 2 * col));
      const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vl + r1 * ROWV + 2 * col));
      bf16x8 vb;
#pragma unroll
      for (int j = 0; j < 4; ++j) { vb[j] = v0[j]; vb[4 + j] = v1[j]; }
#pragma unroll
      for (int i = 0; i < 4; ++i) o[n][i] *= a_i[i];
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, vb, o[n], 0, 0, 0);
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vb, o[n], 0, 0, 0);
    }
  }
  l_run = lane_sum<16>(l_run);
  l_run = lane_sum<32>(l_run);
  if (g4 == 0) {
    ml[wave][li][0] = m_run;
    ml[wave][li][1] = l_run;
  }
  wave_lds_sync();
  float* mine = reinterpret_cast<float*>(vl);     // 16 rows of DK floats fit in 32 rows of DK + 8 bf16
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * g4 + i < R) {
#pragma unroll
      for (int n = 0; n < NVB; ++n) mine[(4 * g4 + i) * DK + 16 * n + li] = o[n][i];
    }
  __syncthreads();
  for (int idx = tid; idx < R * DK; idx += 64 * NW) {
    const int r = idx / DK, d = idx - r * DK, h = g * R + r;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[w][r][0]);
    float a = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = ml[w][r][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[w][r][0] - M);
      a += f * reinterpret_cast<const float*>(vrows[w])[idx];
      l += f * ml[w][r][1];
    }
    if (nsplit == 1) {
      float y = a / l;
      if (gate != nullptr)
        y *= 1.f / (1.f + expf(-bf2f(gate[(size_t)t * ldg + (gate_ph ? (size_t)h : (size_t)h * DK + d)])));
      out[(size_t)t * H * DK + (size_t)h * DK + d] = f2bf(y);
    } else {
      const size_t rec = ((size_t)t * H + h) * nsplit + split;
      pacc[rec * DK + d] = a;
      if (d == 0) {
        pml[rec * 2] = M * LN2;                   // -inf and 0 for a split without keys
        pml[rec * 2 + 1] = l;
      }
    }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" int k8s_window_kv_write(void* kcache, void* vcache, void* qkv, long ld, int koff, int voff, const void* qb,
                                   const void* kb, const void* vb, const float* cos_sin, const int* positions,
                                   const int* slot_mapping, const float* vfirst_in, float* vfirst_out, float lam, int T,
                                   int H, int G, int D, int V, int dims, float eps, int unit, int half_layout,
                                   const void* qnw, const void* knw, const void* hqw, const void* hkw, int f32,
                                   hipStream_t s) {
  if (T <= 0) return 0;
  // G == 0: a layer that attends another layer's cache prepares its queries only
  if (H <= 0 || G < 0 || (G > 0 && H % G) || D <= 0 || D > 512 || V <= 0 || dims < 0 || dims > D || (dims & 1)) return -1;
  if (G > 0 && (kcache == nullptr || vcache == nullptr)) return -1;
  if (dims > 0 && cos_sin == nullptr) return -1;
  if (half_layout && !unit && qnw == nullptr && knw == nullptr && hqw == nullptr && hkw == nullptr && vfirst_in == nullptr &&
      vfirst_out == nullptr && D % 4 == 0 && V % 4 == 0 && dims % 8 == 0 && ld % 4 == 0 && koff % 4 == 0 && voff % 4 == 0 &&
      ((uintptr_t)qkv | (uintptr_t)kcache | (uintptr_t)vcache | (uintptr_t)qb | (uintptr_t)kb | (uintptr_t)vb) %
              (f32 ? 16 : 8) == 0 && (uintptr_t)cos_sin % 16 == 0) {
    const int n = (H + G) * (dims / 8 + (D - dims) / 4) + G * V / 4, ny = (n + 255) / 256;
    const dim3 grid(T, T >= 512 ? 1 : (ny < 65535 ? ny : 65535));
    if (f32)
      rotate_kv_write_kernel<float><<<grid, 256, 0, s>>>((float*)kcache, (float*)vcache, (float*)qkv, ld, koff, voff,
                                                         (const float*)qb, (const float*)kb, (const float*)vb, cos_sin,
                                                         positions, slot_mapping, H, G, D, V, dims);
    else
      rotate_kv_write_kernel<bf16_t><<<grid, 256, 0, s>>>((bf16_t*)kcache, (bf16_t*)vcache, (bf16_t*)qkv, ld, koff, voff,
                                                          (const bf16_t*)qb, (const bf16_t*)kb, (const bf16_t*)vb, cos_sin,
                                                          positions, slot_mapping, H, G, D, V, dims);
    return (int)hipGetLastError();
  }
  const size_t lds = (size_t)4 * D * sizeof(float);
#define K8S_WKW(TA)                                                                                                   \
  window_kv_write_kernel<TA><<<T, 256, lds, s>>>((TA*)kcache, (TA*)vcache, (TA*)qkv, ld, koff, voff, (const TA*)qb,    \
                                                 (const TA*)kb, (const TA*)vb, cos_sin, positions, slot_mapping,      \
                                                 vfirst_in, vfirst_out, lam, H, G, D, V, dims, eps, unit, half_layout, \
                                                 (const TA*)qnw, (const TA*)knw, (const TA*)hqw, (const TA*)hkw)
  if (f32) K8S_WKW(float);
  else K8S_WKW(bf16_t);
#undef K8S_WKW
  return (int)hipGetLastError();
}

extern "C" int k8s_window_pool(float* kpool, float* vpool, const void* kcache, const void* vcache,
                               const int* block_tables, int max_blocks, const int* tok_seq, const int* positions, int T,
                               int G, int D, int V, int P, int bs, int f32, hipStream_t s) {
  if (T <= 0 || P <= 0) return 0;
  if (G <= 0 || D <= 0 || V <= 0 || bs <= 0) return -1;
  const int ppb = (bs + P - 1) / P;
  const int slices = (G * (D + V) + 255) / 256;
  const dim3 grid(T, slices < 16 ? slices : 16);
  if (f32)
    window_pool_kernel<float><<<grid, 256, 0, s>>>(kpool, vpool, (const float*)kcache, (const float*)vcache,
                                                   block_tables, max_blocks, tok_seq, positions, G, D, V, P, bs, ppb);
  else
    window_pool_kernel<bf16_t><<<grid, 256, 0, s>>>(kpool, vpool, (const bf16_t*)kcache, (const bf16_t*)vcache,
                                                    block_tables, max_blocks, tok_seq, positions, G, D, V, P, bs, ppb);
  return (int)hipGetLastError();
}

// Tile rows of the plain kernel for these sizes (0: they do not fit) -- the caller sizes the key splits with it.
extern "C" int k8s_window_tile_rows(int H, int G, int D, int V) {
  if (G <= 0 || H % G) return 0;
  const int R = H / G, nw = R < 8 ? R : 8;
  // LDS floats: KB (D + 1 + V) tile + nw D queries + KB row offsets (2 floats each), within 60 KB
  int KB = (15360 - nw * D - 2) / (D + 1 + V + 2);
  return KB > 64 ? 64 : (KB < 1 ? 0 : KB);
}

// nsplit > 1: pacc [T, H, nsplit, V] and pml [T, H, nsplit, 2] fp32 workspaces.
extern "C" int k8s_window_attention(void* out, float* pacc, float* pml, const void* q, long ldq, const void* gate,
                                    long ldg, const void* kcache, const void* vcache, const float* kpool,
                                    const float* vpool, const int* block_tables, int max_blocks, const int* tok_seq,
                                    const int* positions, int T, int H, int G, int D, int V, int window, int P,
                                    float scale, int sink, int bs, int nsplit, int chunk, float softcap,
                                    const float* sinkv, int gate_ph, const float* slopes, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (H <= 0 || G <= 0 || H % G || D <= 0 || V <= 0 || V > 256 || bs <= 0 || G > 65535) return -1;
  if (window > 0 && P > 0 && (kpool == nullptr || vpool == nullptr || slopes != nullptr)) return -1;
  if (nsplit < 1 || nsplit > 64 || (nsplit > 1 && (pacc == nullptr || pml == nullptr))) return -1;
  const int R = H / G;
  const int nw = R < 8 ? R : 8;
  const int KB = k8s_window_tile_rows(H, G, D, V);
  if (KB < 1) return -2;
  const size_t lds = ((size_t)KB * (D + 1 + V) + (size_t)nw * D + 2 + 2 * (size_t)KB) * sizeof(float);
  const int ppb = P > 0 ? (bs + P - 1) / P : 1;
  const int nacc = (V + 63) / 64;
  const bool vec = D % 8 == 0 && V % 8 == 0 && (f32 || ((long)G * D) % 8 == 0);
#define K8S_WA(TA, NA, VEC)                                                                                           \
  window_attention_kernel<TA, NA, VEC><<<dim3(T, G, nsplit), nw * 64, lds, s>>>(                                      \
      (TA*)out, pacc, pml, (const TA*)q, ldq, (const TA*)gate, ldg, (const TA*)kcache, (const TA*)vcache, kpool,      \
      vpool, block_tables, max_blocks, tok_seq, positions, H, G, D, V, window, P, scale, sink, bs, ppb, KB, nsplit,   \
      chunk, softcap, sinkv, gate_ph, slopes)
#define K8S_WA_V(TA, NA)            \
  do {                              \
    if (vec) K8S_WA(TA, NA, true);  \
    else K8S_WA(TA, NA, false);     \
  } while (0)
#define K8S_WA_T(TA)                     \
  do {                                   \
    if (nacc <= 1) K8S_WA_V(TA, 1);      \
    else if (nacc <= 2) K8S_WA_V(TA, 2); \
    else K8S_WA_V(TA, 4);                \
  } while (0)
  if (f32) K8S_WA_T(float);
  else K8S_WA_T(bf16_t);
#undef K8S_WA_T
#undef K8S_WA_V
#undef K8S_WA
  if (nsplit > 1) {
    if (f32)
      window_merge_kernel<float><<<dim3(T, H), 64, 0, s>>>((float*)out, pacc, pml, (const float*)gate, ldg, positions, H,
                                                           V, nsplit, gate_ph);
    else
      window_merge_kernel<bf16_t><<<dim3(T, H), 64, 0, s>>>((bf16_t*)out, pacc, pml, (const bf16_t*)gate, ldg,
                                                            positions, H, V, nsplit, gate_ph);
  }
  return (int)hipGetLastError();
}

// Whether window_token_kernel takes these sizes.
extern "C" int k8s_window_token_ok(int H, int G, int D, int V, int bs) {
  return G > 0 && H % G == 0 && H / G <= 16 && D == V && (D == 64 || D == 96 || D == 128) && bs > 0 && (bs & (bs - 1)) == 0;
}

// bf16 tokens one by one, each against its visible keys (no pooled blocks); nsplit > 1: pacc [T, H, nsplit, D] and pml
// [T, H, nsplit, 2] fp32 workspaces.
extern "C" int k8s_window_token(void* out, float* pacc, float* pml, const void* q, long ldq, const void* gate, long ldg,
                                const void* kcache, const void* vcache, const int* block_tables, int max_blocks,
                                const int* tok_seq, const int* positions, int T, int H, int G, int D, int window, float scale,
                                int sink, int bs, int nsplit, int chunk, float softcap, const float* sinkv, int gate_ph,
                                const float* slopes, hipStream_t s) {
  if (T <= 0) return 0;
  if (!k8s_window_token_ok(H, G, D, D, bs) || G > 65535 || ldq % 8 || ((uintptr_t)q & 15)) return -1;
  if (nsplit < 1 || nsplit > 64 || (nsplit > 1 && (pacc == nullptr || pml == nullptr))) return -1;
  int bshift = 0;
  while ((1 << bshift) < bs) ++bshift;
#define K8S_WT(DK, NW, AHEAD)                                                                                             \
  window_token_kernel<DK, NW, AHEAD><<<dim3(T, G, nsplit), 64 * NW, 0, s>>>(                                              \
      (bf16_t*)out, pacc, pml, (const bf16_t*)q, ldq, (const bf16_t*)gate, ldg, (const bf16_t*)kcache,                    \
      (const bf16_t*)vcache, block_tables, max_blocks, tok_seq, positions, H, G, window, scale, sink, bshift, nsplit, chunk, \
      softcap, sinkv, gate_ph, slopes)
#define K8S_WT_D(NW, AHEAD)                  \
  do {                                       \
    if (D == 64) K8S_WT(64, NW, AHEAD);      \
    else if (D == 96) K8S_WT(96, NW, AHEAD); \
    else K8S_WT(128, NW, AHEAD);             \
  } while (0)
  // 8 waves while every workgroup runs at once (two on a CU at 64 dimensions, one at more), else 4, of which two to four share a
  // CU.  16 heads over 4 of 128, us, 8 / 4 waves: 64 tokens behind 40 6.2 / 6.6, behind 1000 29 / 36; 66 9.6 / 7.1, 39 / 40; 128 10.4 /
  // 7.9, 53 / 50; of 64, 128 tokens 6.5 / 5.9, 28 / 31, 144 6.7 / 6.5, 35 / 34.  (T x G alone decides: the splits are made for it.)
  if ((long)T * G <= (nsplit > 1 ? 64 : 128)) K8S_WT_D(8, true);
  else if ((long)T * G <= (D == 64 ? 512 : 256)) K8S_WT_D(8, false);
  else K8S_WT_D(4, false);
#undef K8S_WT_D
#undef K8S_WT
  if (nsplit > 1)
    window_merge_kernel<bf16_t><<<dim3(T, H), 64, 0, s>>>((bf16_t*)out, pacc, pml, (const bf16_t*)gate, ldg, positions, H, D,
                                                          nsplit, gate_ph);
  return (int)hipGetLastError();
}

// Whether the matrix-core kernel takes these sizes (else the caller uses k8s_window_attention).
extern "C" int k8s_window_mfma_ok(int H, int G, int D, int V) {
  if (G <= 0 || H % G) return 0;
  const int R = H / G;
  return (R == 1 || R == 2 || R == 4 || R == 8 || R == 16) && D % 8 == 0 && V % 16 == 0 && D <= 256 && V <= 256;
}

// Tokens that one workgroup of window_prompt_kernel takes (0: it does not take these sizes).
extern "C" int k8s_window_prompt_tile(int H, int G, int D, int V, int P, int bs) {
  if (!k8s_window_mfma_ok(H, G, D, V) || P > 0 || D != V || (D != 64 && D != 96 && D != 128) || bs <= 0 || (bs & (bs - 1)))
    return 0;
  return 4 * (16 / (H / G));
}

// Prompt portions in bf16: nseq sequences of at most max_qlen tokens (T in all), cu_q their query offsets.  nsplit > 1 (only
// where k8s_window_prompt_tile > 0): pacc [T, H, nsplit, V] and pml [T, H, nsplit, 2] fp32 workspaces.
extern "C" int k8s_window_attention_mfma(void* out, float* pacc, float* pml, const void* q, long ldq, const void* gate,
                                         long ldg, const void* kcache, const void* vcache, const float* kpool, const float* vpool,
                                         const int* block_tables, int max_blocks, const int* cu_q, const int* positions,
                                         int nseq, int max_qlen, int T, int H, int G, int D, int V, int window, int P,
                                         float scale, int sink, int bs, int nsplit, int chunk, float softcap,
                                         const float* sinkv, int gate_ph, const float* slopes, hipStream_t s) {
  if (nseq <= 0 || max_qlen <= 0) return 0;
  if (nsplit < 1 || nsplit > 64 || (nsplit > 1 && (pacc == nullptr || pml == nullptr || T <= 0))) return -1;
  if (!k8s_window_mfma_ok(H, G, D, V) || bs <= 0 || nseq > 65535 || G > 65535 || ldq % 8 || ((uintptr_t)q & 15)) return -1;
  if (window > 0 && P > 0 && (kpool == nullptr || vpool == nullptr || slopes != nullptr)) return -1;
  const int R = H / G, ppb = P > 0 ? (bs + P - 1) / P : 1;
  if (k8s_window_prompt_tile(H, G, D, V, P, bs) > 0) {
    const int tpb = k8s_window_prompt_tile(H, G, D, V, P, bs);
    const dim3 grid((max_qlen + tpb - 1) / tpb * nsplit, G, nseq);
    int bshift = 0;
    while ((1 << bshift) < bs) ++bshift;
    const size_t stage = (size_t)2 * 64 * (D + 8 + V + 8) * 2;                     // two buffers of 64 rows
    const size_t merge = (size_t)4 * 64 * (4 * (V / 16) + 2) * sizeof(float);   // one group's results
    const size_t lds = stage > merge ? stage : merge;
#define K8S_WP(DK, SPLIT)                                                                                               \
  do {                                                                                                                  \
    static bool grown = false;   /* more LDS than a launch gets by default */                                           \
    if (!grown) {                                                                                                       \
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(window_prompt_kernel<DK, DK, SPLIT>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                   \
      if (e != hipSuccess) return (int)e;                                                                               \
      grown = true;                                                                                                     \
    }                                                                                                                   \
    window_prompt_kernel<DK, DK, SPLIT><<<grid, 512, lds, s>>>(                                                    \
        (bf16_t*)out, pacc, pml, (const bf16_t*)q, ldq, (const bf16_t*)gate, ldg, (const bf16_t*)kcache,                \
        (const bf16_t*)vcache, block_tables, max_blocks, cu_q, positions, H, G, window, scale, sink, bshift, nsplit, R, \
        chunk, softcap, sinkv, gate_ph, slopes);                                                                        \
  } while (0)
#define K8S_WP_D(SPLIT)                \
  do {                                 \
    if (D == 64) K8S_WP(64, SPLIT);    \
    else if (D == 96) K8S_WP(96, SPLIT); \
    else K8S_WP(128, SPLIT);           \
  } while (0)
    if (nsplit > 1) K8S_WP_D(true);
    else K8S_WP_D(false);
#undef K8S_WP_D
#undef K8S_WP
    if (nsplit > 1)
      window_merge_kernel<bf16_t><<<dim3(T, H), 64, 0, s>>>((bf16_t*)out, pacc, pml, (const bf16_t*)gate, ldg, positions, H,
                                                            V, nsplit, gate_ph);
    return (int)hipGetLastError();
  }
  if (nsplit > 1) return -1;
  const size_t lds = (size_t)32 * ((D + 8) + (V + 8)) * 2;
  constexpr int NCB = 2;
  const int TPB = 4 * NCB * (16 / R);
  const dim3 grid((max_qlen + TPB - 1) / TPB, G, nseq);
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cus = n;
  }
  const bool pf = (long)grid.x * grid.y * grid.z <= cus;
#define K8S_WM_P(NKK, NVB, PF)                                                                                        \
  window_attention_mfma_kernel<NKK, NVB, NCB, PF><<<grid, 256, lds, s>>>(                                             \
      (bf16_t*)out, (const bf16_t*)q, ldq, (const bf16_t*)gate, ldg, (const bf16_t*)kcache, (const bf16_t*)vcache,    \
      kpool, vpool, block_tables, max_blocks, cu_q, positions, H, G, D, V, window, P, scale, sink, bs, ppb, R, chunk, \
      softcap, sinkv, gate_ph, slopes)
#define K8S_WM(NKK, NVB)               \
  do {                                 \
    if (pf) K8S_WM_P(NKK, NVB, true);  \
    else K8S_WM_P(NKK, NVB, false);    \
  } while (0)
  if (D <= 64 && V <= 64) K8S_WM(2, 4);
  else if (D <= 128 && V <= 128) K8S_WM(4, 8);
  else K8S_WM_P(8, 16, false);
#undef K8S_WM
#undef K8S_WM_P
  return (int)hipGetLastError();
}
