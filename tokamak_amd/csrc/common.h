// Shared device helpers for the gfx950 kernels: bf16 storage conversions,
// 64-lane wave reductions, launch-error reporting.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tk {

typedef uint16_t bf16_t;  // raw bfloat16 bits; arithmetic is always done in float

__device__ __forceinline__ float bf16_to_float(bf16_t v) {
  return __uint_as_float(static_cast<uint32_t>(v) << 16);
}

// round-to-nearest-even; NaN stays NaN.  gfx950 converts in hardware
// (v_cvt_pk_bf16_f32), which the compiler emits for these casts.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const f32x2_t f = {lo, hi};
  const bf16x2_t v = __builtin_convertvector(f, bf16x2_t);
  return *reinterpret_cast<const uint32_t*>(&v);
}

__device__ __forceinline__ bf16_t float_to_bf16(float f) {
  return static_cast<bf16_t>(pack_bf16x2(f, 0.f) & 0xffffu);
}

template <typename T> struct Elem;
template <> struct Elem<float> {
  static __device__ __forceinline__ float load(const float* p) { return *p; }
  static __device__ __forceinline__ void store(float* p, float v) { *p = v; }
};
template <> struct Elem<bf16_t> {
  static __device__ __forceinline__ float load(const bf16_t* p) { return bf16_to_float(*p); }
  static __device__ __forceinline__ void store(bf16_t* p, float v) { *p = float_to_bf16(v); }
};

// Four consecutive elements p[0..3] of which the first `valid` exist.  `wide`: p is 16-byte
// (float32) or 8-byte (bfloat16) aligned, so four that all exist go out as one store: a
// wave's 4-byte stores of an MFMA result tile are sixteen scattered pieces per row of it and
// cost a product of 64 rows a fifth of its time.
template <typename T>
__device__ __forceinline__ void store_four(T* p, float a, float b, float c, float d, int valid, bool wide);
template <>
__device__ __forceinline__ void store_four<float>(float* p, float a, float b, float c, float d, int valid, bool wide) {
  if (wide && valid >= 4) {
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
    return;
  }
  if (valid > 0) p[0] = a;
  if (valid > 1) p[1] = b;
  if (valid > 2) p[2] = c;
  if (valid > 3) p[3] = d;
}
template <>
__device__ __forceinline__ void store_four<bf16_t>(bf16_t* p, float a, float b, float c, float d, int valid, bool wide) {
  if (wide && valid >= 4) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(a, b), pack_bf16x2(c, d));
    return;
  }
  if (valid > 0) p[0] = float_to_bf16(a);
  if (valid > 1) p[1] = float_to_bf16(b);
  if (valid > 2) p[2] = float_to_bf16(c);
  if (valid > 3) p[3] = float_to_bf16(d);
}
// Whether rows of `ld` elements starting at p keep every fourth element aligned for store_four.
template <typename T>
__device__ __forceinline__ bool rows_take_wide_stores(const T* p, long ld) {
  return (reinterpret_cast<uintptr_t>(p) % (4 * sizeof(T))) == 0 && ld % 4 == 0;
}

constexpr int kWave = 64;

// Exchanges between lanes by the vector unit's own lane paths (__shfl_xor goes through LDS: some 100 cycles a level,
// these 8 to 16; a reduction over the wave six levels).
//
// The value of the lane whose number differs in bit 0 or 1 (level 0, 1).  Levels 2 and 3 take the mirrored lane of eight
// and of sixteen: it lies in the other four, the other eight, whose lanes all hold the same after the levels before.
template <int LEVEL>
__device__ __forceinline__ uint32_t lane_other(uint32_t v) {
  static_assert(LEVEL >= 0 && LEVEL < 4, "levels 4 and 5 come as pairs");
  constexpr int kControl = LEVEL == 0 ? 0xB1 /* quad_perm 1 0 3 2 */ : LEVEL == 1 ? 0x4E /* quad_perm 2 3 0 1 */
                           : LEVEL == 2 ? 0x141 /* row_half_mirror */ : 0x140 /* row_mirror */;
  return __builtin_amdgcn_update_dpp(0u, v, kControl, 0xf, 0xf, false);
}
template <int LEVEL>
__device__ __forceinline__ float lane_other(float v) { return __uint_as_float(lane_other<LEVEL>(__float_as_uint(v))); }

// Lanes l and l ^ 16 (l ^ 32): both get the pair (value of the lane without that bit, value of the lane with it).
struct LanePair {
  uint32_t first, second;
  __device__ __forceinline__ float a() const { return __uint_as_float(first); }
  __device__ __forceinline__ float b() const { return __uint_as_float(second); }
};
__device__ __forceinline__ LanePair pair16(uint32_t v) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return {r[0], r[1]};
}
__device__ __forceinline__ LanePair pair32(uint32_t v) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return {r[0], r[1]};
}
// v of lane l with v of lane l ^ 16, and over all four lanes l, l ^ 16, l ^ 32, l ^ 48: the same bits in each of them
__device__ __forceinline__ float sum16(float v) { const LanePair p = pair16(__float_as_uint(v)); return p.a() + p.b(); }
__device__ __forceinline__ float sum32(float v) { const LanePair p = pair32(__float_as_uint(v)); return p.a() + p.b(); }
__device__ __forceinline__ float max16(float v) { const LanePair p = pair16(__float_as_uint(v)); return fmaxf(p.a(), p.b()); }
__device__ __forceinline__ float max32(float v) { const LanePair p = pair32(__float_as_uint(v)); return fmaxf(p.a(), p.b()); }

// The value of lane l ^ D.
template <int D>
__device__ __forceinline__ float lane_xor(float v) {
  static_assert(D == 1 || D == 2 || D == 4 || D == 8 || D == 16 || D == 32, "a bit of the lane's number");
  const uint32_t u = __float_as_uint(v);
  if constexpr (D <= 2) return __uint_as_float(lane_other<D - 1>(u));
  if constexpr (D == 4)      // the mirrored lane of eight, then the mirrored one of four
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, lane_other<2>(u), 0x1B /* quad_perm 3 2 1 0 */, 0xf, 0xf, false));
  if constexpr (D == 8) return __uint_as_float(__builtin_amdgcn_update_dpp(0u, u, 0x128 /* row_ror:8 */, 0xf, 0xf, false));
  const LanePair p = D == 16 ? pair16(u) : pair32(u);
  return threadIdx.x & D ? p.a() : p.b();      // (blocks are rows of threads in this library: the lane's number is threadIdx.x % 64)
}
// The sum over the lanes whose numbers differ in bits FROM, 2 FROM, ..., below TO.
template <int FROM, int TO>
__device__ __forceinline__ float sum_lanes(float v) {
  if constexpr (FROM >= TO) return v;
  else if constexpr (FROM == 16) return sum_lanes<32, TO>(sum16(v));
  else if constexpr (FROM == 32) return sum32(v);
  else return sum_lanes<FROM * 2, TO>(v + lane_xor<FROM>(v));
}

// (all lanes get the same bits: a level's two addends are the same two numbers in each of its lanes)
__device__ __forceinline__ float wave_sum(float v) {
  v += lane_other<0>(v);
  v += lane_other<1>(v);
  v += lane_other<2>(v);
  v += lane_other<3>(v);
  return sum32(sum16(v));
}

// Orders one wave's LDS accesses (a wave's LDS instructions execute in order; this
// keeps the compiler from moving them across the point).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, lane_other<0>(v));
  v = fmaxf(v, lane_other<1>(v));
  v = fmaxf(v, lane_other<2>(v));
  v = fmaxf(v, lane_other<3>(v));
  return max32(max16(v));
}

// The best (value, index) of the wave in every lane; take(value, at, other value, its index) keeps the better of two, whichever
// of them comes first.
template <typename Take>
__device__ __forceinline__ void wave_best(float& value, int& at, const Take& take) {
  take(value, at, lane_other<0>(value), (int)lane_other<0>((uint32_t)at));
  take(value, at, lane_other<1>(value), (int)lane_other<1>((uint32_t)at));
  take(value, at, lane_other<2>(value), (int)lane_other<2>((uint32_t)at));
  take(value, at, lane_other<3>(value), (int)lane_other<3>((uint32_t)at));
  LanePair v = pair16(__float_as_uint(value)), i = pair16((uint32_t)at);
  value = v.a();
  at = (int)i.first;
  take(value, at, v.b(), (int)i.second);
  v = pair32(__float_as_uint(value));
  i = pair32((uint32_t)at);
  value = v.a();
  at = (int)i.first;
  take(value, at, v.b(), (int)i.second);
}

// Sum over a block of up to 1024 threads; `scratch` holds >= 16 floats of LDS.
// Every thread of the block must call it; all get the result.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int nwaves = (blockDim.x + kWave - 1) / kWave;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nwaves; ++i) t += scratch[i];
  return t;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  v = wave_max(v);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int nwaves = (blockDim.x + kWave - 1) / kWave;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = scratch[0];
  for (int i = 1; i < nwaves; ++i) t = fmaxf(t, scratch[i]);
  return t;
}

inline int launch_status() { return static_cast<int>(hipGetLastError()); }

}  // namespace tk

#define TK_API extern "C" __attribute__((visibility("default")))
