// The Gated DeltaNet token for 16-bit state pools (fp16, bf16), on the matrix
// cores. fp32 pools run gdn_tile.h's VALU token.
//
// Both contractions of a token with the stored state, kv = S^T k_hat and
// sq = S^T q_hat, are one matrix product: S (128 rows x the columns) against a
// handful of vectors. The state is 16-bit, so it is an operand of
// v_mfma_f32_16x16x32_{f16,bf16} as it lies in the registers, with no
// conversion; k_hat and q_hat, which are fp32, are split into 16-bit parts that
// sum to them:
//   fp16 pool: 1024 x = hi + lo, hi = fp16(1024 x), lo = fp16(1024 x - hi):
//              22 to 24 of x's 24 bits (at most one fp32 unit of x off; |x| <= 1,
//              and the 1024 keeps lo clear of fp16's subnormals);
//   bf16 pool: x = hi + mid + lo, each part the bf16 rounding of what is left:
//              all 24 bits.
// Every part x state product is exact in fp32, and the MFMA adds 32 of them
// with fewer roundings than the fma chains that this replaces (measured, error
// of a 32-term sum against 64 bits over the sum of magnitudes: 1.2e-8 rms
// fp16, 0.8e-8 bf16; four fma chains of eight 1.6e-8 and 0.8e-8).
//
// The readout follows from the old state: S' = alpha S + k_hat delta gives
//   y = (S'^T q_hat) * scale = (alpha sq + delta (k_hat . q_hat)) * scale,
// so a token touches the state once for both products, and per element the
// VALU is left with the update (a product, an fma, half a packed conversion)
// where the chains took two fmas more.
//
// Lane map. Operand element e of lane (g = l / 16, n = l % 16) is row
// 32 w + g + 4 e of column n, e = 0..7: the rows that lane group g of a decode
// wave holds (gdn_tile.h, LaneMap), so a decode lane feeds its own registers.
// The other operand holds the parts: row m of its 16 rows is part m % 4, so
// every lane's four results are parts 0..3 of its column, and all lane groups
// hold the same sums: no cross-lane step is left within a wave.
//
// Fixed order (defines the bits, the same in decode and prefill): one MFMA
// (two for bf16) per row block w of 32 rows from a zero accumulator, its parts
// combined smallest first, then the blocks as (w0 + w1) + (w2 + w3).
#pragma once

#include "gdn_tile.h"

namespace braid {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The 16-bit parts of a normalised vector pair (k_hat, q_hat) and the MFMAs
// over them. kParts: parts of both vectors; kFrags: MFMAs per row block;
// part_of(f, m): the part in row m (mod 4) of MFMA f's operand.
template <class Tag>
struct Parts;

template <>
struct Parts<F16> {
  static constexpr int kParts = 4;  // k hi, k lo, q hi, q lo
  static constexpr int kQ = 2;      // q's first part
  static constexpr int kSplit = 2;
  static constexpr int kFrags = 1;
  __device__ __forceinline__ static int part_of(int, int m) { return m & 3; }
  // The vectors are held scaled by this, a power of two.
  static constexpr float kScale = 1024.f;
  // Two scaled values' parts, packed (x0 in the low halves). x - hi is exact.
  __device__ __forceinline__ static void split2(float x0, float x1, uint32_t (&p)[kSplit]) {
    p[0] = pack_f16x2(x0, x1);
    p[1] = pack_f16x2(x0 - f16_widen(p[0] & 0xffffu), x1 - f16_widen(p[0] >> 16));
  }
  __device__ __forceinline__ static f32x4v mfma(u32x4 a, u32x4 b) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b),
                                                  (f32x4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  }
  __device__ __forceinline__ static float kv(const f32x4v (&d)[kFrags]) {
    return d[0][1] + d[0][0];
  }
  __device__ __forceinline__ static float sq(const f32x4v (&d)[kFrags]) {
    return d[0][3] + d[0][2];
  }
};

template <>
struct Parts<BF16> {
  static constexpr int kParts = 6;  // k hi, mid, lo, q hi, mid, lo
  static constexpr int kQ = 3;
  static constexpr int kSplit = 3;
  static constexpr int kFrags = 2;
  // MFMA 0: k hi, k mid, k lo, q hi; MFMA 1: q mid, q lo (twice).
  __device__ __forceinline__ static int part_of(int f, int m) {
    return f == 0 ? (m & 3) : 4 + (m & 1);
  }
  static constexpr float kScale = 1.f;
  __device__ __forceinline__ static void split2(float x0, float x1, uint32_t (&p)[kSplit]) {
#pragma unroll
    for (int i = 0; i < kSplit; ++i) {
      p[i] = pack_bf16x2(x0, x1);
      x0 -= bf16_widen(p[i] & 0xffffu);
      x1 -= bf16_widen(p[i] >> 16);
    }
  }
  __device__ __forceinline__ static f32x4v mfma(u32x4 a, u32x4 b) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b),
                                                   (f32x4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  }
  __device__ __forceinline__ static float kv(const f32x4v (&d)[kFrags]) {
    return (d[0][2] + d[0][1]) + d[0][0];
  }
  __device__ __forceinline__ static float sq(const f32x4v (&d)[kFrags]) {
    return (d[1][1] + d[1][0]) + d[0][3];
  }
};

// A 16-bit pool element pair's halves, widened.
template <class Tag>
__device__ __forceinline__ float half_of(uint32_t pair, int h) {
  const uint32_t b = h ? pair >> 16 : pair & 0xffffu;
  if constexpr (std::is_same<Tag, F16>::value) return f16_widen(b);
  else return bf16_widen(b);
}
template <class Tag>
__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  if constexpr (std::is_same<Tag, F16>::value) return pack_f16x2(lo, hi);
  else return pack_bf16x2(lo, hi);
}

// delta and y from the products with the scaled vectors: alpha_s = alpha /
// kScale (exact), kq = k_hat . q_hat.
__device__ __forceinline__ float delta_of(float v, float alpha_s, float beta, float kv) {
  return (v - alpha_s * kv) * beta;
}
__device__ __forceinline__ float readout_of(float alpha_s, float sq, float delta, float kq) {
  return fmaf(alpha_s, sq, delta * kq) * kYScale;
}

// ---------------------------------------------------------------------------
// Decode.

// One wave's row block of the normalised q and k, in the order its lanes read
// them: part[p][g][i / 2] holds rows 32 w + g + 4 i and + 4 (i + 1) (i even) of
// part p, packed; k[g][i] the fp32 k_hat of row 32 w + g + 4 i.
template <class Tag>
struct QKParts {
  alignas(16) uint16_t part[Parts<Tag>::kParts][kRowGroups][kRowsPerLane];
  alignas(16) float k[kRowGroups][kRowsPerLane];
};

// A decode lane's operands: its row block's parts and its rows' k_hat, and
// k_hat . q_hat.
template <class Tag>
struct QKOps {
  u32x4 a[Parts<Tag>::kFrags];
  float kh[kRowsPerLane];
  float kq;
};

// From the pairs every lane of the wave holds (elements 2 lane, 2 lane + 1):
// the norms and the dot product by the wave butterfly; the 16 lanes that hold
// the wave's row block write it to the wave's own LDS copy, and every lane
// reads its operands back (no workgroup barrier: only this wave touches buf).
template <class Tag, class LM>
__device__ __forceinline__ void split_qk_lds(const LM& L, float2 q2, float2 k2, QKParts<Tag>& buf,
                                             QKOps<Tag>& out) {
  using P = Parts<Tag>;
  const float qi = inv_norm(q2), ki = inv_norm(k2);
  const float2 qh = make_float2(q2.x * qi, q2.y * qi), kh = make_float2(k2.x * ki, k2.y * ki);
  if (L.rg == L.w) {
    // Rows 2 cc and 2 cc + 1 of the block: row groups g0 and g0 + 1, index i.
    const int g0 = (2 * L.cc) & 3, i = L.cc >> 1;
    uint32_t pk[P::kSplit], pq[P::kSplit];
    P::split2(kh.x * P::kScale, kh.y * P::kScale, pk);
    P::split2(qh.x * P::kScale, qh.y * P::kScale, pq);
#pragma unroll
    for (int p = 0; p < P::kSplit; ++p) {
      buf.part[p][g0][i] = (uint16_t)pk[p];
      buf.part[p][g0 + 1][i] = (uint16_t)(pk[p] >> 16);
      buf.part[P::kQ + p][g0][i] = (uint16_t)pq[p];
      buf.part[P::kQ + p][g0 + 1][i] = (uint16_t)(pq[p] >> 16);
    }
    buf.k[g0][i] = kh.x;
    buf.k[g0 + 1][i] = kh.y;
  }
  // The reads below take values other lanes of this wave wrote (see
  // normalize_qk_lds).
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // Behind the writes: the readout alone needs it.
  out.kq = wave_sum(kh.x * qh.x + kh.y * qh.y);
#pragma unroll
  for (int f = 0; f < P::kFrags; ++f)
    out.a[f] = *reinterpret_cast<const u32x4*>(&buf.part[P::part_of(f, L.cc)][L.rg][0]);
  loadN<kRowsPerLane>(&buf.k[L.rg][0], out.kh);
}

// Column partials of the four row blocks, and the token's gates.
struct TileLds16 {
  float kv[kWaves][kHD];
  float sq[kWaves][kHD];
  float gate[2];  // this token's alpha, beta (publish_gates)
};

// One decode token on this lane's 8 x CPL block: the products with the stored
// state, one exchange across the waves, delta and the update (each new element
// rounded to fp32, then narrowed). Contains the token's one workgroup barrier.
// The caller stores the state, then reads out (token16_readout): a conditional
// readout ahead of the stores lets the compiler copy the stores into both of
// its branches, and a wave then writes each row in two parts.
template <class Tag, int CPL>
__device__ __forceinline__ void gdn_token16(const LaneMap<CPL>& L, Row<Tag, CPL> (&S)[kRowsPerLane],
                                            const QKOps<Tag>& qk, const float (&v)[CPL],
                                            TileLds16& lds, float (&delta)[CPL]) {
  using P = Parts<Tag>;
  float kv[CPL], sq[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    // Column c's eight rows, two to a register.
    u32x4 b;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t r0 = S[2 * m].raw[c >> 1], r1 = S[2 * m + 1].raw[c >> 1];
      b[m] = __builtin_amdgcn_perm(r1, r0, (c & 1) ? 0x07060302u : 0x05040100u);
    }
    f32x4v d[P::kFrags];
#pragma unroll
    for (int f = 0; f < P::kFrags; ++f) d[f] = P::mfma(qk.a[f], b);
    kv[c] = P::kv(d);
    sq[c] = P::sq(d);
  }
  if (L.rg == 0) {
    store_cols(L, lds.kv[L.w], kv);
    store_cols(L, lds.sq[L.w], sq);
  }
  __syncthreads();
  column_sums_take(L, kv, lds.kv);
  const float alpha = lds.gate[0], beta = lds.gate[1], alpha_s = alpha * (1.f / P::kScale);
#pragma unroll
  for (int c = 0; c < CPL; ++c) delta[c] = delta_of(v[c], alpha_s, beta, kv[c]);
#pragma unroll
  for (int i = 0; i < kRowsPerLane; ++i) {
#pragma unroll
    for (int c = 0; c < CPL; c += 2) {
      const float n0 = fmaf(alpha, S[i].get(c), qk.kh[i] * delta[c]);
      const float n1 = fmaf(alpha, S[i].get(c + 1), qk.kh[i] * delta[c + 1]);
      S[i].set2(c, n0, n1);
    }
  }
}

// The outputs of the lanes that store them, into the tile's y row.
template <class Tag, int CPL>
__device__ __forceinline__ void token16_readout(const LaneMap<CPL>& L, const QKOps<Tag>& qk,
                                                TileLds16& lds, const float (&delta)[CPL],
                                                float* y_row) {
  if (!L.stores_y()) return;
  float sq[CPL], y[CPL];
  column_sums_take(L, sq, lds.sq);
  const float alpha_s = lds.gate[0] * (1.f / Parts<Tag>::kScale);
#pragma unroll
  for (int c = 0; c < CPL; ++c) y[c] = readout_of(alpha_s, sq[c], delta[c], qk.kq);
  store_cols(L, y_row, y);
}

}  // namespace braid
