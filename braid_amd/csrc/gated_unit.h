// One (token, value head) unit of the gated RMSNorm readout, shared by the
// readout kernel (gated_norm.hip) and the fused decode step (gdn_scan.hip), so
// both compute the same bits. See gated_norm.hip for the arithmetic.
#pragma once

#include "quant_common.h"

namespace braid {
namespace quant {
namespace {

constexpr int kUnit = 128;                          // HD
constexpr int kLanesPerUnit = 32;                   // 4 elements per lane
constexpr int kUnitsPerBlock = (kThreads / 64) * 2;  // two units per wave

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Act-dtype narrowing of two fp32 values, round to nearest even, returned both
// packed (for the store) and widened back (for the arithmetic that follows).
// The packed vector conversion consumes the already-rounded fp32 operands; a
// scalar `(_Float16)(a * b)` may be contracted into one mixed-precision op
// that rounds the exact product once, straight to 16 bits.
template <class Tag>
struct Narrow;
template <>
struct Narrow<XF32> {
  __device__ __forceinline__ static void pair(float& a, float& b, uint32_t&) {}
};
template <>
struct Narrow<XF16> {
  __device__ __forceinline__ static void pair(float& a, float& b, uint32_t& bits) {
    const f16x2 h = __builtin_convertvector((f32x2){a, b}, f16x2);
    bits = __builtin_bit_cast(uint32_t, h);
    a = (float)h[0];
    b = (float)h[1];
  }
};
template <>
struct Narrow<XBF16> {
  __device__ __forceinline__ static void pair(float& a, float& b, uint32_t& bits) {
    bits = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
    a = __uint_as_float(bits << 16);
    b = __uint_as_float(bits & 0xffff0000u);
  }
};

// Four consecutive elements at p + i (i a multiple of 4, 16/8-byte aligned).
__device__ __forceinline__ void load4(XF32, const float* p, long i, float (&o)[4]) {
  const f32x4 v = *reinterpret_cast<const f32x4*>(p + i);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = v[e];
}
template <class Tag>
__device__ __forceinline__ void load4(Tag tag, const uint16_t* p, long i, float (&o)[4]) {
  const u32x2 r = *reinterpret_cast<const u32x2*>(p + i);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = widen(tag, (uint16_t)((r[e >> 1] >> (16 * (e & 1))) & 0xffffu));
}

// Rounds o[0..3] to the act dtype in place and stores them at p + i. Plain
// (cacheable) stores: the quantize pass reads core back right away, and at
// prefill sizes it then comes from the Infinity Cache (4073 tokens: 42.6 ->
// 41.2 us for the readout against nontemporal stores).
__device__ __forceinline__ void round_store4(XF32, float* p, long i, float (&o)[4]) {
  *reinterpret_cast<f32x4*>(p + i) = (f32x4){o[0], o[1], o[2], o[3]};
}
template <class Tag>
__device__ __forceinline__ void round_store4(Tag, uint16_t* p, long i, float (&o)[4]) {
  uint32_t r0, r1;
  Narrow<Tag>::pair(o[0], o[1], r0);
  Narrow<Tag>::pair(o[2], o[3], r1);
  *reinterpret_cast<u32x2*>(p + i) = (u32x2){r0, r1};
}
template <class Tag>
__device__ __forceinline__ void round4(Tag, float (&o)[4]) {
  uint32_t unused;
  Narrow<Tag>::pair(o[0], o[1], unused);
  Narrow<Tag>::pair(o[2], o[3], unused);
}

// One unit's computation from its loaded y (c, widened) and z values: writes
// core and folds |core| into the running max m.
template <class ATag>
__device__ __forceinline__ void gated_unit(float (&c)[4], const float (&zf)[4], const f32x4& gm,
                                           float eps, bool live, typename ATag::T* core, long i,
                                           float& m) {
  round4(ATag{}, c);
  float ss = (c[0] * c[0] + c[1] * c[1]) + (c[2] * c[2] + c[3] * c[3]);
  static_assert(kLanesPerUnit == 32, "a unit's sum runs over lane bits 0-4");
  ss += lane_xor<1>(ss);
  ss += lane_xor<2>(ss);
  ss += lane_xor<4>(ss);
  ss += lane_xor<8>(ss);
  ss += lane_xor<16>(ss);
  const float r = rsqrtf(ss * (1.0f / kUnit) + eps);  // mean: exact power-of-two scale
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = c[e] * r;
  round4(ATag{}, o);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float h = gm[e] * o[e];
    const float s = zf[e] / (1.0f + expf(-zf[e]));
    o[e] = h * s;
  }
  if (live) {
    round_store4(ATag{}, core, i, o);
#pragma unroll
    for (int e = 0; e < 4; ++e) m = nan_max(m, fabsf(o[e]));
  }
}

// The same unit on 16 lanes, eight consecutive elements each: a lane adds its two
// quads, which the 32-lane butterfly's first stage adds across lanes, and the
// other stages follow at half the distance, so the bits are gated_unit's.
template <class ATag>
__device__ __forceinline__ void gated_unit_wide(float (&c)[kVec], const float (&zf)[kVec],
                                                const float (&gm)[kVec], float eps, bool live,
                                                typename ATag::T* core, long i, float& m) {
  uint32_t bits[kVec / 2];
#pragma unroll
  for (int e = 0; e < kVec; e += 2) Narrow<ATag>::pair(c[e], c[e + 1], bits[e / 2]);
  float ss = ((c[0] * c[0] + c[1] * c[1]) + (c[2] * c[2] + c[3] * c[3])) +
             ((c[4] * c[4] + c[5] * c[5]) + (c[6] * c[6] + c[7] * c[7]));
  ss += lane_xor<1>(ss);
  ss += lane_xor<2>(ss);
  ss += lane_xor<4>(ss);
  ss += lane_xor<8>(ss);
  const float r = rsqrtf(ss * (1.0f / kUnit) + eps);
  float o[kVec];
#pragma unroll
  for (int e = 0; e < kVec; ++e) o[e] = c[e] * r;
#pragma unroll
  for (int e = 0; e < kVec; e += 2) Narrow<ATag>::pair(o[e], o[e + 1], bits[e / 2]);
#pragma unroll
  for (int e = 0; e < kVec; ++e) {
    const float h = gm[e] * o[e];
    const float s = zf[e] / (1.0f + expf(-zf[e]));
    o[e] = h * s;
  }
  if (live) {
#pragma unroll
    for (int e = 0; e < kVec; e += 2) Narrow<ATag>::pair(o[e], o[e + 1], bits[e / 2]);
    if constexpr (sizeof(typename ATag::T) == 2) {
      *reinterpret_cast<u32x4*>(core + i) = (u32x4){bits[0], bits[1], bits[2], bits[3]};
    } else {
      *reinterpret_cast<f32x4*>(core + i) = (f32x4){o[0], o[1], o[2], o[3]};
      *reinterpret_cast<f32x4*>(core + i + 4) = (f32x4){o[4], o[5], o[6], o[7]};
    }
#pragma unroll
    for (int e = 0; e < kVec; ++e) m = nan_max(m, fabsf(o[e]));
  }
}

}  // namespace
}  // namespace quant
}  // namespace braid
