// Per-head RMSNorm and rotary embedding of rows held by lane groups, shared
// by the decode kernels' prologue and the prompt pass.
#pragma once

#include "common.hpp"

namespace asrattn {
namespace {

template <typename T>
__device__ __forceinline__ void unpack(const uint4& r, float* out);

template <>
__device__ __forceinline__ void unpack<float>(const uint4& r, float* out) {
  out[0] = __uint_as_float(r.x); out[1] = __uint_as_float(r.y);
  out[2] = __uint_as_float(r.z); out[3] = __uint_as_float(r.w);
}

template <>
__device__ __forceinline__ void unpack<bf16_raw>(const uint4& r, float* out) {
  out[0] = bf16_lo(r.x); out[1] = bf16_hi(r.x);
  out[2] = bf16_lo(r.y); out[3] = bf16_hi(r.y);
  out[4] = bf16_lo(r.z); out[5] = bf16_hi(r.z);
  out[6] = bf16_lo(r.w); out[7] = bf16_hi(r.w);
}

template <typename T>
__device__ __forceinline__ uint4 pack(const float* x);

template <>
__device__ __forceinline__ uint4 pack<float>(const float* x) {
  return make_uint4(__float_as_uint(x[0]), __float_as_uint(x[1]), __float_as_uint(x[2]), __float_as_uint(x[3]));
}

template <>
__device__ __forceinline__ uint4 pack<bf16_raw>(const float* x) {
  return make_uint4(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]), pack_bf16x2(x[6], x[7]));
}

// x rounded to T (and back): where the reference's element-wise ops round.
template <typename T>
__device__ __forceinline__ float round_to(float x) {
  if constexpr (sizeof(T) == 2) return bf16_to_f32(f32_to_bf16(x));
  return x;
}

// The same for two values (one conversion instruction in bf16).
template <typename T>
__device__ __forceinline__ void round_pair(float& a, float& b) {
  if constexpr (sizeof(T) == 2) {
    const uint32_t u = pack_bf16x2(a, b);
    a = bf16_lo(u);
    b = bf16_hi(u);
  }
}

// The values of lane l ^ (LPK / 2): a row rotation for 16-lane rows, else
// through the LDS crossbar.
template <int LPK>
__device__ __forceinline__ float half_row_partner(float x) {
  if constexpr (LPK == 16)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xF, 0xF, false));  // row_ror:8
  return __shfl_xor(x, LPK / 2, 64);
}

// Per-head RMSNorm and rotary embedding of one row slice -- lane `sub` of
// the LPK lanes holding a head_dim row, EPL elements -- in the reference's
// rounding order (qwen3_asr.py:322-330): the norm x * rsqrt(mean(x^2) +
// eps) * w in fp32, rounded once; the rotation x c + r s with r = (-x[d/2:],
// x[:d/2]) rounded after each product and after the sum.  Element e of lane
// sub pairs with element e of lane sub ^ LPK/2.  w, cs and sn are the
// lane's slices of the weights and tables (loaded by the caller).  norm,
// weighted and rotated say what this row gets (uniform over its lanes);
// any_norm and any_rot whether any row of the launch does (uniform over the
// grid).  All lanes of the wave must take part.
template <typename T, int HD, int LPK>
__device__ __forceinline__ uint4 prologue_row(uint4 raw, bool any_norm, bool norm, bool weighted, const uint4& w,
                                              bool any_rot, bool rotated, const uint4& cs, const uint4& sn, float eps,
                                              int sub) {
  constexpr int EPL = Elem<T>::kPerVec;
  float x[EPL];
  unpack<T>(raw, x);
  if (any_norm) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) ss = fmaf(x[e], x[e], ss);
    ss = group_sum<LPK>(ss);
    const float r = rsqrtf(ss * (1.f / HD) + eps);
    float wv[EPL];
    unpack<T>(w, wv);
#pragma unroll
    for (int e = 0; e < EPL; e += 2) {
      float a = weighted ? x[e] * r * wv[e] : x[e] * r;
      float b = weighted ? x[e + 1] * r * wv[e + 1] : x[e + 1] * r;
      round_pair<T>(a, b);
      x[e] = norm ? a : x[e];
      x[e + 1] = norm ? b : x[e + 1];
    }
  }
  if (any_rot) {
    float cv[EPL], sv[EPL];
    unpack<T>(cs, cv);
    unpack<T>(sn, sv);
    const bool lower = sub < LPK / 2;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float partner = half_row_partner<LPK>(x[e]);
      float a = x[e] * cv[e], b = (lower ? -partner : partner) * sv[e];
      round_pair<T>(a, b);
      x[e] = rotated ? a + b : x[e];
    }
  }
  return pack<T>(x);
}

}  // namespace
}  // namespace asrattn
