// Shared device helpers for the gfx950 (MI355X, CDNA4) kernels.
// Wave = 64 lanes everywhere; bf16 tensors are moved as 16-byte vectors (8 x bf16).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include <stdint.h>

namespace k8sllm {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef uint16_t bf16_t;  // raw storage type on the host/ABI side

constexpr int WAVE = 64;

__device__ __forceinline__ float bf2f(bf16_t v) { return __uint_as_float(((uint32_t)v) << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) {
  __bf16 b = (__bf16)f;  // v_cvt_pk_bf16_f32 (RNE, NaN-preserving) on gfx950
  return __builtin_bit_cast(bf16_t, b);
}
// Unpack 2 bf16 held in one dword.
__device__ __forceinline__ float lo_bf(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_bf(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) {
  return (uint32_t)f2bf(a) | ((uint32_t)f2bf(b) << 16);
}

// Element load / store as fp32 for kernels templated on the storage type (bf16 or true fp32).
template <typename T> __device__ __forceinline__ float ldf(const T* p, size_t i);
template <> __device__ __forceinline__ float ldf<float>(const float* p, size_t i) { return p[i]; }
template <> __device__ __forceinline__ float ldf<bf16_t>(const bf16_t* p, size_t i) { return bf2f(p[i]); }
template <typename T> __device__ __forceinline__ void stf(T* p, size_t i, float v);
template <> __device__ __forceinline__ void stf<float>(float* p, size_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void stf<bf16_t>(bf16_t* p, size_t i, float v) { p[i] = f2bf(v); }

// The value of lane ^ O, and sums and maxima over the two, by register moves: a shuffle goes through LDS and its address
// (a wave sum in a chain of them 187 -> 55 ns).  Every lane of the wave takes part.  Same operands as by shuffles, so the same results.
template <int O>
__device__ __forceinline__ float lane_xor(float v) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8, "within rows of 16 lanes");
  const auto move = [](float x, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  if constexpr (O == 1) return move(v, std::integral_constant<int, 0xB1>{});          // quad_perm 1 0 3 2
  else if constexpr (O == 2) return move(v, std::integral_constant<int, 0x4E>{});     // quad_perm 2 3 0 1
  else if constexpr (O == 8) return move(v, std::integral_constant<int, 0x128>{});    // row_ror 8
  else return move(move(v, std::integral_constant<int, 0x141>{}), std::integral_constant<int, 0x1B>{});  // mirrored in 8, then in 4
}
// (a of the lanes without bit O, b of those with it) and the same of lane ^ O: the two halves exchange the other's operand
template <int O>
__device__ __forceinline__ void lane_swap(float a, float b, float& x, float& y) {
  static_assert(O == 16 || O == 32, "rows of 16 lanes");
  if constexpr (O == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    x = __uint_as_float(r[0]), y = __uint_as_float(r[1]);
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    x = __uint_as_float(r[0]), y = __uint_as_float(r[1]);
  }
}
template <int O>
__device__ __forceinline__ float lane_sum(float v) {
  if constexpr (O >= 16) {
    float x, y;
    lane_swap<O>(v, v, x, y);
    return x + y;
  } else {
    return v + lane_xor<O>(v);
  }
}
template <int O>
__device__ __forceinline__ float lane_max(float v) {
  if constexpr (O >= 16) {
    float x, y;
    lane_swap<O>(v, v, x, y);
    return fmaxf(x, y);
  } else {
    return fmaxf(v, lane_xor<O>(v));
  }
}
__device__ __forceinline__ float wave_sum(float v) {
  return lane_sum<1>(lane_sum<2>(lane_sum<4>(lane_sum<8>(lane_sum<16>(lane_sum<32>(v))))));
}
__device__ __forceinline__ float wave_max(float v) {
  return lane_max<1>(lane_max<2>(lane_max<4>(lane_max<8>(lane_max<16>(lane_max<32>(v))))));
}

// OCP MX e4m3 (K16 block-scaled activations; fp8.hip has the format): one E8M0 byte per 32 values, the smallest
// power of two >= max|block| / 448 (127 for an all-zero block, clamped to [1, 253]), and the exact reciprocal.
__device__ __forceinline__ uint32_t mx_e8m0(float amax) {
  const uint32_t b = __float_as_uint(amax * (1.f / 448.f));
  uint32_t e = (b >> 23) + ((b & 0x7fffffu) != 0u);
  if (amax == 0.f) e = 127u;
  return min(max(e, 1u), 253u);
}
__device__ __forceinline__ float mx_inv_scale(uint32_t e) { return __uint_as_float((254u - e) << 23); }
// 4 fp32 values x inv -> 4 e4m3 bytes (one dword), saturated, round-to-nearest-even
__device__ __forceinline__ uint32_t mx_pack4(float a, float b, float c, float d, float inv) {
  auto cl = [&](float t) { return fminf(fmaxf(t * inv, -448.f), 448.f); };
  int p = __builtin_amdgcn_cvt_pk_fp8_f32(cl(a), cl(b), 0, false);
  p = __builtin_amdgcn_cvt_pk_fp8_f32(cl(c), cl(d), p, true);
  return (uint32_t)p;
}
// bf16 rounding of an fp32 value (MX producers quantize the bf16 value the bf16 path would have stored)
__device__ __forceinline__ float bf_round(float f) { return bf2f(f2bf(f)); }
// Byte offset of the E8M0 scale of 32-value block kb of row m in an [M][K] MX tensor.  Layout [K / 128][M][4]: the
// four scales of a 128-value k-tile of a row form one dword, and the dwords of consecutive rows are adjacent -- so a
// GEMM stages one k-tile's scales for a run of rows as one contiguous LDS-DMA (one cache line per 32 rows, not one
// per row).
__device__ __forceinline__ size_t mx_scale_off(size_t m, int kb, int M) {
  return ((size_t)(kb >> 2) * (size_t)M + m) * 4 + (size_t)(kb & 3);
}
// MX store of one value per lane, the 32 lanes of an aligned half-wave holding one block (row m, columns col..,
// col of the half-wave's first lane a multiple of 32): shuffle max, then one e4m3 byte per lane and the block's E8M0.
__device__ __forceinline__ void mx_store_lane(uint8_t* oq, uint8_t* oe, size_t m, int col, int K, int M, float v) {
  const float amax = lane_max<16>(lane_max<8>(lane_max<4>(lane_max<2>(lane_max<1>(fabsf(v))))));
  const uint32_t e = mx_e8m0(amax);
  oq[m * (size_t)K + col] = (uint8_t)(mx_pack4(v, 0.f, 0.f, 0.f, mx_inv_scale(e)) & 0xffu);
  if ((col & 31) == 0) oe[mx_scale_off(m, col >> 5, M)] = (uint8_t)e;
}

// Four consecutive elements as fp32, and back; pointers aligned to the four elements.
template <typename T> __device__ __forceinline__ f32x4 ldf4(const T* p);
template <> __device__ __forceinline__ f32x4 ldf4<float>(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
template <> __device__ __forceinline__ f32x4 ldf4<bf16_t>(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return f32x4{lo_bf(u.x), hi_bf(u.x), lo_bf(u.y), hi_bf(u.y)};
}
template <typename T> __device__ __forceinline__ void stf4(T* p, f32x4 v);
template <> __device__ __forceinline__ void stf4<float>(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
template <> __device__ __forceinline__ void stf4<bf16_t>(bf16_t* p, f32x4 v) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
}

// Block-wide sum for blockDim.x <= 1024; `red` must hold >= 16 floats of LDS.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = (lane < nw) ? red[lane] : 0.f;
  t = wave_sum(t);
  __syncthreads();
  return t;
}

// Workgroup barrier that waits for this wave's LDS traffic only: __syncthreads() also drains the outstanding global
// loads, which would put the prefetched inputs of the next tokens back on the recurrence's latency chain.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0); vmcnt and expcnt untouched
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The sum over a workgroup of 4 full waves, in every thread: 16 lanes by register moves, the rows of a wave by lane reads, the
// waves through 4 floats of `red` (of which every call of a kernel has its own) behind a barrier that waits for LDS only.  The
// row norms are a chain of latencies: block_sum's 12 shuffles and its waits for the stores in flight cost one row of 2048 0.3 us
// (3.45 -> 3.16), a norm on both sides 0.65 (4.29 -> 3.64), 2048 rows 0.3 - 0.8 of 5.4 - 10.7.
template <int CTRL>
__device__ __forceinline__ float lane_add(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row_total(float v, float* red) {
  v = lane_add<0x140>(lane_add<0x141>(lane_add<0x4E>(lane_add<0xB1>(v))));     // lanes ^ 1, ^ 2, mirrored in 8, in 16
  const auto lane = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l)); };
  const float w = (lane(0) + lane(16)) + (lane(32) + lane(48));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  lds_barrier();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Chunk g of a varlen batch cut into chunks of Lc tokens per sequence: (sequence, chunk in the sequence, chunks of the
// sequence), or sequence -1 when g is past the last chunk.  Idle (position < 0) and empty sequences have no chunks.
struct WkvChunk { int s, c, n; };
__device__ __forceinline__ WkvChunk wkv_find_chunk(int g, const int* cu_q, const int* positions, int nseq, int Lc) {
  for (int s = 0; s < nseq; ++s) {
    const int a = cu_q[s], len = cu_q[s + 1] - a;
    const int n = (len > 0 && positions[a] >= 0) ? (len + Lc - 1) / Lc : 0;
    if (g < n) return WkvChunk{s, g, n};
    g -= n;
  }
  return WkvChunk{-1, 0, 0};
}

// 32-bit mixing hash (murmur3 finalizer) used for counter-based RNG and deterministic init.
__device__ __forceinline__ uint32_t fmix32(uint32_t h) {
  h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
  return h;
}
__device__ __forceinline__ uint32_t hash3(uint32_t a, uint32_t b, uint32_t c) {
  return fmix32(a ^ fmix32(b + 0x9e3779b9u ^ fmix32(c + 0x7f4a7c15u)));
}
// Uniform in (0, 1): 24 random bits, never 0.
__device__ __forceinline__ float u01(uint32_t h) { return ((h >> 8) + 0.5f) * (1.0f / 16777216.0f); }

// ---- checked builds (python -m k8s_llm_scheduler_amd._build --checked -> ops/_C_checked*.so, loaded with
// K8S_CHECKED=1): every index a kernel derives from DATA (block tables, slot mappings, token ids, context lengths) is
// range-checked before it addresses memory.  A violation is recorded in a device record the host reads after each
// engine step (ops.check_read) and the index is clamped to a valid one, so the kernel finishes without touching
// memory it does not own -- the bounds-assert debug build of SURVEY.md section 5 (race detection / sanitizers), with
// no trap: a trapping kernel would take the device down for every process on it.  Release builds compile none of it.
struct K8sCheck {
  unsigned count;         // violations since the last reset
  unsigned code, line;    // the first one: check code (K8S_CHK_*), source line
  unsigned unit;          // translation unit (K8S_CHK_UNIT_*)
  long long value;        // the offending value
  long long kv_slots;     // bounds, set by the host: KV-cache slots (blocks x block size)
  long long num_blocks;   // KV-cache blocks
  long long vocab;        // embedding rows
};
enum { K8S_CHK_SLOT = 1, K8S_CHK_BLOCK = 2, K8S_CHK_CTX = 3, K8S_CHK_TOKEN = 4 };

}  // namespace k8sllm

#ifdef K8S_CHECKED
// One record pointer per translation unit (kernels are built without relocatable device code); K8S_CHECK_UNIT
// defines the unit's bind function, k8s_check_bind (bindings) points every unit at the same record.
static __device__ k8sllm::K8sCheck* g_k8s_check;
__device__ __forceinline__ static void k8s_check_fail(unsigned unit, unsigned code, unsigned line, long long v) {
  k8sllm::K8sCheck* c = g_k8s_check;
  if (c == nullptr) return;
  // the record is written with vector memory instructions only: the address is forced into VGPRs
  unsigned long long a = reinterpret_cast<unsigned long long>(c);
  asm volatile("" : "+v"(a));
  k8sllm::K8sCheck* cv = reinterpret_cast<k8sllm::K8sCheck*>(a);
  const unsigned old = __hip_atomic_fetch_add(&cv->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (old == 0) {
    __hip_atomic_store(&cv->code, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&cv->line, line, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&cv->unit, unit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&cv->value, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}
__device__ __forceinline__ static long long k8s_bound(int code) {
  const k8sllm::K8sCheck* c = g_k8s_check;
  if (c == nullptr) return 0x7fffffffffffffffLL;
  return code == k8sllm::K8S_CHK_SLOT ? c->kv_slots : code == k8sllm::K8S_CHK_BLOCK ? c->num_blocks : c->vocab;
}
// var must lie in [lo, bound(code)); otherwise record it and set var = fallback
#define K8S_CHECK_RANGE(var, lo, code, fallback)                                          \
  do {                                                                                    \
    if ((long long)(var) < (long long)(lo) || (long long)(var) >= k8s_bound(code)) {      \
      k8s_check_fail(K8S_CHK_THIS_UNIT, (code), __LINE__, (long long)(var));              \
      (var) = (fallback);                                                                 \
    }                                                                                     \
  } while (0)
// var must be <= maxv (a bound the kernel knows itself); otherwise record it and set var = maxv
#define K8S_CHECK_MAX(var, maxv, code)                                                    \
  do {                                                                                    \
    if ((long long)(var) > (long long)(maxv)) {                                           \
      k8s_check_fail(K8S_CHK_THIS_UNIT, (code), __LINE__, (long long)(var));              \
      (var) = (maxv);                                                                     \
    }                                                                                     \
  } while (0)
// a condition that must hold (no clamp: the caller handles the failure)
#define K8S_CHECK_TRUE(cond, code, value)                                                 \
  do {                                                                                    \
    if (!(cond)) k8s_check_fail(K8S_CHK_THIS_UNIT, (code), __LINE__, (long long)(value)); \
  } while (0)
#define K8S_CHECK_UNIT(name)                                                              \
  extern "C" int k8s_check_bind_##name(void* rec) {                                       \
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_k8s_check), &rec, sizeof(rec));            \
  }
#else
#define K8S_CHECK_RANGE(var, lo, code, fallback) \
  do {                                           \
  } while (0)
#define K8S_CHECK_TRUE(cond, code, value) \
  do {                                    \
  } while (0)
#define K8S_CHECK_MAX(var, maxv, code) \
  do {                                 \
  } while (0)
#define K8S_CHECK_UNIT(name) \
  extern "C" int k8s_check_bind_##name(void*) { return -1; }
#endif

#define K8S_CHECK_LAUNCH() (void)hipGetLastError()
