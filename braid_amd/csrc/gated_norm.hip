// Gated RMSNorm readout of the GDN mixer, fused with the out_proj input's
// dynamic FP8 quantization.
//
// Reference behaviour (braid/model/gdn.py:373-387 `_readout`, braid/model/
// norm.py:48-71 `rms_norm_gated`, then braid/model/quant.py:209-229 on the
// result): for each (token, value head) unit of HD = 128 scan outputs y,
//   c    = y.to(act)                         scan output cast to the act dtype
//   xf   = c * rsqrt(mean(c^2) + eps)       F.rms_norm in fp32, no weight
//   h    = gamma * xf.to(act)                gamma fp32 [HD]; promotes to fp32
//   o    = h * silu(z.float())               silu(x) = x / (1 + exp(-x))
//   core = o.to(act)                         the out_proj input [N, H*HD]
// and, when the out_proj weight is FP8, (q, scale) = quantize_act(core) over
// the whole [N, H*HD] tensor.
//
// Launch 1 (gated_norm_amax) computes `core` and, in the same pass, one
// NaN-propagating partial max of |core| per block: it replaces the amax pass of
// the quantizer, so the readout and the quantization together are the same two
// launches as the quantization alone. Launch 2 is the quantizer's own second
// pass, reading `core` back (bf16: 2 B per element, L2/MALL-resident at
// decode sizes).
//
// Layout: a wave takes two units per iteration, 32 lanes each, four
// consecutive elements per lane (16-byte fp32 loads of y, 8-byte loads of z).
// The sum of squares is an in-lane pair sum followed by a 32-lane butterfly,
// so both halves of the wave reduce independently. The reduction order differs
// from torch's rms_norm kernel: the result agrees to fp32 rounding before the
// act-dtype casts (gated by tolerance, not bits).
#include "gated_unit.h"

namespace braid {
namespace {

using namespace quant;

// YTag: dtype of the scan output y (fp32, or already the act dtype). ATag: the
// act dtype of z and core. Each wave iteration takes one pair of units, one
// per half-wave. (Two pairs per iteration, loaded before either is computed,
// measured 3% slower at 4073 tokens, four 8%: more bytes in flight per wave
// did not pay for the registers and the longer iteration.)
template <class YTag, class ATag>
__global__ void __launch_bounds__(kThreads)
gated_norm_amax(const typename YTag::T* __restrict__ y, const typename ATag::T* __restrict__ z,
                const float* __restrict__ gamma, float eps, long units,
                typename ATag::T* __restrict__ core, float* __restrict__ partial) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane / kLanesPerUnit, sub = lane % kLanesPerUnit;
  const f32x4 gm = *reinterpret_cast<const f32x4*>(gamma + 4 * sub);
  float m = 0.f;
  const long step = (long)gridDim.x * kUnitsPerBlock;
  // Both halves of a wave run every iteration (the butterfly needs all 64
  // lanes); a half past the end works on zeros and stores nothing.
  for (long u0 = ((long)blockIdx.x * (kThreads / 64) + wave) * 2; u0 < units; u0 += step) {
    const long u = u0 + half;
    const bool live = u < units;
    const long i = u * kUnit + 4 * sub;
    float c[4] = {0.f, 0.f, 0.f, 0.f}, zz[4] = {0.f, 0.f, 0.f, 0.f};
    if (live) {
      load4(YTag{}, y, i, c);
      load4(ATag{}, z, i, zz);
    }
    gated_unit<ATag>(c, zz, gm, eps, live, core, i, m);
  }
  m = block_nan_max(m);
  if (partial != nullptr && threadIdx.x == 0) partial[blockIdx.x] = m;
}

// The same for large inputs, four units per wave iteration, 16 lanes each with
// 16-byte accesses of 16-bit elements: a grid of kMaxBlocks leaves 16 waves on a
// CU, and their bytes in flight set the rate once y and z come from HBM. The same
// bits (gated_unit_wide). 6,888 tokens, bf16 y, cold: 54.1 -> 46.0 us (3.7 TB/s),
// 4,073 34.1 -> 30.4, 1,024 10.3 -> 9.6, 512 6.7 -> 6.6; below that the narrow
// kernel spreads the units over more CUs.
template <class YTag, class ATag>
__global__ void __launch_bounds__(kThreads)
gated_norm_amax_wide(const typename YTag::T* __restrict__ y,
                     const typename ATag::T* __restrict__ z, const float* __restrict__ gamma,
                     float eps, long units, typename ATag::T* __restrict__ core,
                     float* __restrict__ partial) {
  constexpr int kLanes = kUnit / kVec, kPerWave = 64 / kLanes;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane / kLanes, sub = lane % kLanes;
  float gm[kVec];
  load_vec(XF32{}, gamma, kVec * sub, gm);
  float m = 0.f;
  const long step = (long)gridDim.x * (kThreads / 64) * kPerWave;
  // All lanes run every iteration (the butterfly needs them); units past the
  // end work on zeros and store nothing.
  for (long u0 = ((long)blockIdx.x * (kThreads / 64) + wave) * kPerWave; u0 < units; u0 += step) {
    const long u = u0 + row;
    const bool live = u < units;
    const long i = u * kUnit + kVec * sub;
    float c[kVec], zz[kVec];
    if (live) {
      load_vec(YTag{}, y, i, c);
      load_vec(ATag{}, z, i, zz);
    } else {
#pragma unroll
      for (int e = 0; e < kVec; ++e) c[e] = zz[e] = 0.f;
    }
    gated_unit_wide<ATag>(c, zz, gm, eps, live, core, i, m);
  }
  m = block_nan_max(m);
  if (partial != nullptr && threadIdx.x == 0) partial[blockIdx.x] = m;
}

constexpr int64_t kWideUnits = 16384;

int norm_blocks(int64_t units) {
  const int64_t want = (units + kUnitsPerBlock - 1) / kUnitsPerBlock;
  return (int)(want < 1 ? 1 : (want > kMaxBlocks ? kMaxBlocks : want));
}

template <class YTag, class ATag>
int launch(const void* yv, const void* zv, const float* gamma, float eps, int64_t units,
           void* corev, uint8_t* q, float* scale, float* partial, hipStream_t stream) {
  using AT = typename ATag::T;
  const auto* y = static_cast<const typename YTag::T*>(yv);
  const auto* z = static_cast<const AT*>(zv);
  AT* core = static_cast<AT*>(corev);
  const int blocks = norm_blocks(units);
  auto* const kern =
      units >= kWideUnits ? gated_norm_amax_wide<YTag, ATag> : gated_norm_amax<YTag, ATag>;
  kern<<<blocks, kThreads, 0, stream>>>(y, z, gamma, eps, units, core,
                                        q != nullptr ? partial : nullptr);
  if (q != nullptr) {
    const int64_t n = units * kUnit;
    const int vec = ((reinterpret_cast<uintptr_t>(q) & 7u) == 0) ? 1 : 0;
    quantize<ATag><<<blocks_for(n), kThreads, 0, stream>>>(core, partial, blocks, scale, q, n, vec);
  }
  const int st = hip_status(hipGetLastError(), "launching gated_rmsnorm kernels");
  return st != BRAID_OK ? st : ok();
}

template <class ATag>
int dispatch_y(int y_dtype, const void* y, const void* z, const float* gamma, float eps,
               int64_t units, void* core, uint8_t* q, float* scale, float* partial,
               hipStream_t stream, int act_dtype) {
  if (y_dtype == BRAID_F32)
    return launch<XF32, ATag>(y, z, gamma, eps, units, core, q, scale, partial, stream);
  if (y_dtype == act_dtype)
    return launch<ATag, ATag>(y, z, gamma, eps, units, core, q, scale, partial, stream);
  return fail(BRAID_EINVAL, "y must be fp32 or the activation dtype");
}

}  // namespace
}  // namespace braid

using namespace braid;

extern "C" int braid_gated_rmsnorm_workspace(int64_t units) { return norm_blocks(units); }

extern "C" int braid_gated_rmsnorm_quant(const void* y, int y_dtype, const void* z,
                                         int act_dtype, const float* gamma, float eps,
                                         int64_t units, int HD, void* core, uint8_t* q,
                                         float* scale, float* partial, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (HD != kUnit) return fail(BRAID_EINVAL, "head_dim must be 128, got " + std::to_string(HD));
  if (units < 0) return fail(BRAID_EINVAL, "negative unit count");
  const bool quant = q != nullptr;
  if (quant && (scale == nullptr || partial == nullptr))
    return fail(BRAID_EINVAL, "q, scale and partial must be given together");
  if (!quant && (scale != nullptr))
    return fail(BRAID_EINVAL, "q, scale and partial must be given together");
  if (quant && units == 0) return fail(BRAID_EINVAL, "x must not be empty");
  if (units == 0) return ok();
  if (y == nullptr || z == nullptr || gamma == nullptr || core == nullptr)
    return fail(BRAID_EINVAL, "y/z/gamma/core must be non-null");
  if (!aligned16(y) || !aligned16(z) || !aligned16(core) || !aligned16(gamma))
    return fail(BRAID_EINVAL, "y, z, gamma and core must be 16-byte aligned");
  switch (act_dtype) {
    case BRAID_F32:
      return dispatch_y<XF32>(y_dtype, y, z, gamma, eps, units, core, q, scale, partial, stream,
                              act_dtype);
    case BRAID_F16:
      return dispatch_y<XF16>(y_dtype, y, z, gamma, eps, units, core, q, scale, partial, stream,
                              act_dtype);
    case BRAID_BF16:
      return dispatch_y<XBF16>(y_dtype, y, z, gamma, eps, units, core, q, scale, partial, stream,
                               act_dtype);
    default: return fail(BRAID_EINVAL, "activation must be fp32, bf16 or fp16");
  }
}
