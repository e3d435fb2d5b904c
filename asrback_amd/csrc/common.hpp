// Device helpers shared by the attention kernels (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "asrattn.h"

namespace asrattn {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();

// bf16 is carried as raw 16-bit storage; the kernels convert explicitly.
using bf16_raw = uint16_t;

__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); }
__device__ __forceinline__ float bf16_to_f32(bf16_raw x) { return __uint_as_float((uint32_t)x << 16); }

// Round-to-nearest-even fp32 -> bf16 pair; gfx950 does this in one
// v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  bf16x2_t r;
  r.x = (__bf16)lo;
  r.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ bf16_raw f32_to_bf16(float x) {
  return (bf16_raw)(pack_bf16x2(x, 0.f) & 0xffffu);
}

// 2^x on the hardware exponential unit (v_exp_f32).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Element type traits: 16-byte vector loads, converted to fp32.
template <typename T>
struct Elem;

template <>
struct Elem<float> {
  static constexpr int kPerVec = 4;  // elements per 16-byte load
  static __device__ __forceinline__ void load16(const float* p, float* out) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
  }
  static __device__ __forceinline__ float load1(const float* p) { return *p; }
  static __device__ __forceinline__ void store1(float* p, float x) { *p = x; }
};

template <>
struct Elem<bf16_raw> {
  static constexpr int kPerVec = 8;
  static __device__ __forceinline__ void load16(const bf16_raw* p, float* out) {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    out[0] = bf16_lo(v.x); out[1] = bf16_hi(v.x);
    out[2] = bf16_lo(v.y); out[3] = bf16_hi(v.y);
    out[4] = bf16_lo(v.z); out[5] = bf16_hi(v.z);
    out[6] = bf16_lo(v.w); out[7] = bf16_hi(v.w);
  }
  static __device__ __forceinline__ float load1(const bf16_raw* p) { return bf16_to_f32(*p); }
  static __device__ __forceinline__ void store1(bf16_raw* p, float x) { *p = f32_to_bf16(x); }
};

// The values of lanes l and l ^ OFF as a pair (a, b): a lane whose OFF bit
// is clear gets its own value in a and its partner's in b (the partner gets
// the same two values, in some order).  OFF 16 and 32 are one VALU lane swap
// each (v_permlane16_swap, v_permlane32_swap: rows of 16 lanes, halves of
// 32), OFF 8 a DPP rotation by 8 inside each row, which is l ^ 8; none goes
// through the LDS crossbar as ds_bpermute does.
template <int OFF>
__device__ __forceinline__ void lane_pair(float x, float& a, float& b) {
  static_assert(OFF == 8 || OFF == 16 || OFF == 32, "lane pair offset");
  if constexpr (OFF == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else if constexpr (OFF == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else {
    a = x;
    b = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xF, 0xF, false));  // row_ror:8
  }
}

// Butterfly sum inside aligned groups of W lanes (W a power of two <= 64);
// every lane of the group ends with the group's sum.  Steps within 16 lanes
// use DPP (quad permutes, then half-row and row mirrors, which pair equal
// partial sums once the smaller groups are summed); wider steps are lane
// swaps (lane_pair).
template <int W>
__device__ __forceinline__ float group_sum(float x) {
  if constexpr (W >= 2) x += __builtin_amdgcn_update_dpp(0.f, x, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
  if constexpr (W >= 4) x += __builtin_amdgcn_update_dpp(0.f, x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
  if constexpr (W >= 8) x += __builtin_amdgcn_update_dpp(0.f, x, 0x141, 0xF, 0xF, false);  // row_half_mirror
  if constexpr (W >= 16) x += __builtin_amdgcn_update_dpp(0.f, x, 0x140, 0xF, 0xF, false); // row_mirror
  float a, b;
  if constexpr (W >= 32) {
    lane_pair<16>(x, a, b);
    x = a + b;
  }
  if constexpr (W >= 64) {
    lane_pair<32>(x, a, b);
    x = a + b;
  }
  return x;
}

// Raw buffer resource over [base, base + bytes): 16-byte loads past the end
// return zeros, so guarded loads need no branch.  base must be uniform over
// the wave.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ uint4 buffer_load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset, uint32_t soffset = 0) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, soffset, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// The same load marked nontemporal (cache policy NT): for data read exactly
// once, such as a decoder step's keys and values; it measured 17% more HBM
// throughput on a Qwen3 decode step than the default policy.
__device__ __forceinline__ uint4 buffer_load16_stream(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  constexpr int kNontemporal = 2;  // gfx940+ cache-policy bit NT
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, 0, kNontemporal);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// A load of memory that nothing writes during the launch, at an address
// uniform over the wave: through the scalar cache, also in kernels whose
// atomics make the compiler assume otherwise (it then takes vector loads,
// which wait behind the ones in flight).
template <typename T>
__device__ __forceinline__ T load_uniform(const T* p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) T*>(reinterpret_cast<uintptr_t>(p));
}

// Keys sequence b uses in a decoder step: seqused_k, else positions + 1,
// else all of them; clamped to [0, max_len].
__device__ __forceinline__ int decode_key_count(const int32_t* seqused, const int64_t* positions,
                                                int b, int max_len) {
  long long n = max_len;
  if (seqused != nullptr) {
    n = load_uniform(seqused + b);
  } else if (positions != nullptr) {
    n = load_uniform(positions + b) + 1;
  }
  if (n > max_len) n = max_len;
  if (n < 0) n = 0;
  return (int)n;
}

}  // namespace asrattn
