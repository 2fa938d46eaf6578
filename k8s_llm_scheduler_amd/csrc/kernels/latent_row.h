// A token's row of a latent cache, and its queries' rotation: mixers.hip's latent_kv_write, and stream32.hip's launch that absorbs the
// queries of few tokens beside it.
#pragma once

#include "common.h"

namespace k8sllm {

template <typename TA>
struct LatentRows {
  TA* cache;                // [slots][C + R]
  const TA* dkv;            // [T] rows of C + R, ldd apart
  const TA* normw;
  TA* q;                    // [T][H][Dn + R]
  const float* cos_sin;     // [positions][dims] = cos | sin
  const int* positions;
  const int* slot_mapping;
  int C, R, H, Dn, dims;
  float eps;
  long ldd;
};

// Whether latent_row takes these sizes and places: whole vectors of four elements.
template <typename TA>
inline bool latent_row_ok(const LatentRows<TA>& a) {
  const uintptr_t at = (uintptr_t)a.cache | (uintptr_t)a.dkv | (uintptr_t)a.normw | (uintptr_t)a.q;
  return a.C % 4 == 0 && a.C <= 1024 && a.R % 4 == 0 && a.Dn % 4 == 0 && a.dims % 8 == 0 && a.ldd % 4 == 0 && at % (4 * sizeof(TA)) == 0 &&
         (uintptr_t)a.cos_sin % 16 == 0;
}

// cache[slot] = [rms-norm(dkv[:C]) normw | rotated dkv[C:]], the last R of every head of q rotated in place, by a workgroup of 256; an
// idle row (position < 0) is left alone, a row without a slot has its queries rotated only.  The row, its norm's weight and the queries
// are in flight at once, four elements a thread.  IL: pairs are 2 i, 2 i + 1, otherwise i, i + dims / 2.
template <typename TA, bool IL>
__device__ __forceinline__ void latent_row(const LatentRows<TA>& a, int t, float* red) {
  const int pos = a.positions[t], slot = a.slot_mapping[t];
  const int tid = threadIdx.x, half = a.dims / 2, quads = half / 4;
  const TA* d = a.dkv + (size_t)t * a.ldd;
  const bool in = 4 * tid < a.C;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  const f32x4 x = in ? ldf4(d + 4 * tid) : zero, w = in ? ldf4(a.normw + 4 * tid) : zero;
  if (pos < 0) return;
  const float* cs = a.cos_sin + (size_t)pos * a.dims;
  auto rotate = [&](const TA* from, TA* to, int i) {     // pairs i .. i + 3
    const f32x4 c = ldf4(cs + i), s = ldf4(cs + half + i);
    if (IL) {
      const f32x4 u = ldf4(from + 2 * i), v = ldf4(from + 2 * i + 4);
      stf4(to + 2 * i, f32x4{u[0] * c[0] - u[1] * s[0], u[1] * c[0] + u[0] * s[0], u[2] * c[1] - u[3] * s[1], u[3] * c[1] + u[2] * s[1]});
      stf4(to + 2 * i + 4,
           f32x4{v[0] * c[2] - v[1] * s[2], v[1] * c[2] + v[0] * s[2], v[2] * c[3] - v[3] * s[3], v[3] * c[3] + v[2] * s[3]});
    } else {
      const f32x4 u = ldf4(from + i), v = ldf4(from + half + i);
      f32x4 y, z;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = u[e] * c[e] - v[e] * s[e];
        z[e] = v[e] * c[e] + u[e] * s[e];
      }
      stf4(to + i, y);
      stf4(to + half + i, z);
    }
  };
  TA* row = a.cache + (size_t)max(slot, 0) * (a.C + a.R);
  TA* qt = a.q + (size_t)t * a.H * (a.Dn + a.R);
  // the last piece of work is the row's own rotated part: heads first, so that its threads are others than the row's
  for (int i = 255 - tid; i < (a.H + 1) * quads; i += 256) {
    const int h = i / quads, p = 4 * (i - h * quads);
    if (h < a.H) {
      TA* qh = qt + (size_t)h * (a.Dn + a.R) + a.Dn;
      rotate(qh, qh, p);
    } else if (slot >= 0) {
      rotate(d + a.C, row + a.C, p);
    }
  }
  if (slot >= 0)
    for (int i = a.dims + 4 * tid; i < a.R; i += 1024) stf4(row + a.C + i, ldf4(d + a.C + i));
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) ss += x[e] * x[e];
  const float inv = 1.0f / sqrtf(row_total(ss, red) / (float)a.C + a.eps);
  if (in && slot >= 0) {
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = x[e] * inv * w[e];
    stf4(row + 4 * tid, y);
  }
}

}  // namespace k8sllm
