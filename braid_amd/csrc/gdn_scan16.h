// The chunk prefill scan for 16-bit state pools, on the matrix cores
// (gdn_mfma.h): the tile stays in registers as MFMA operands, a token's kv and
// sq products are four MFMAs a wave, and the update's products k_hat * delta
// are MFMAs too, which leaves the VALU one fma and half a packed conversion
// per state element and token.
//
// What bounds it: VALU issue and the dependent chain of a token (products ->
// delta -> update -> next products) at one or two waves per SIMD.
#pragma once

#include "gdn_mfma.h"

namespace braid {

// Lane geometry. A wave owns kCols columns of one tile, a workgroup kWaves waves'
// columns, a tile is kParts workgroups.
//
// With 16 columns a wave (layouts 1 and 2) lane (g = lane / 16, j = lane % 16)
// holds column j and all four row blocks, and a token takes one state product
// per block. With 8 (layout 4) or 4 columns (layout 8) the lanes of a 16-lane
// row hold a column's row blocks in halves or quarters (h), 2 or 1 blocks a
// lane; the operand's 16 rows then stand for the parts of the 2 or 4 blocks
// that one product covers (block h' in the rows that lane groups g = h' mod
// 4 / kNB receive), so a lane's result is its column's only where g stands for
// its own h, and the others take it over from there (spread16).
template <int Layout>
struct Scan16Map {
  static constexpr int kNB = Layout == 4 ? 2 : (Layout == 8 ? 1 : 4);  // row blocks per lane
  static constexpr int kH = 4 / kNB;                                   // lanes a column is split over
  static constexpr int kCols = 4 * kNB;                                // columns per wave
  static constexpr int kWaves = Layout == 2 ? 8 : 4;   // that run the tokens
  static constexpr int kPrep = 4;                       // that prepare the stages, a round each
  static constexpr int kThreads = 64 * (kWaves + kPrep);
  static constexpr int kParts = kHD / (kWaves * kCols);
  static constexpr int kSlots = 64 / kCols;     // tokens whose y one store instruction covers
  int wave, lane, g, j, h, col, slot;
  __device__ __forceinline__ Scan16Map(int tid) {
    lane = tid & 63;
    wave = tid >> 6;
    g = lane >> 4;
    j = lane & 15;
    h = j / kCols;
    col = wave * kCols + j % kCols;  // the lane's column within the workgroup's
    slot = lane / kCols;
  }
  // Row i of the lane's block s.
  __device__ __forceinline__ int row(int s, int i) const {
    return (kNB * h + s) * kRowsPerWave + g + kRowGroups * i;
  }
  // The block that row m of the operand of the lane's block s stands for.
  __device__ __forceinline__ static int block_of(int s, int m) {
    return kNB * ((m >> 2) & (kH - 1)) + s;
  }
};

// A stage: the next kStage tokens' inputs in LDS, double buffered, so that
// the workgroup meets at one barrier a stage.
//   part  the vectors' 16-bit parts: part p of row 32 w + g + 4 i at word
//         p * kPartRow + w * 16 + g * 4 + i / 2 (two rows i, i + 1 to a word):
//         an operand is one 16-byte read, and the strides keep both the reads
//         (parts and row groups of one block) and the writes (the 16 lanes and
//         four tokens of a wave) on distinct banks.
//   kf    k_hat in fp32, in the order the update's MFMA takes it: row 32 w + g
//         + 4 (4 u + m) at (w / 2) * kKfHalf + (4 g + m) * 4 + (w % 2) * 2 + u.
constexpr int kStage16 = 16;
constexpr int kPartRow = 68;
constexpr int kKfHalf = 68;
constexpr int kKfToken = 144;
constexpr int kGateTokens = 64;  // gates are evaluated 64 tokens at a time, one per lane

template <class Tag, int Layout>
struct alignas(16) Stage16 {
  using LM = Scan16Map<Layout>;
  static constexpr int kPartToken = Parts<Tag>::kParts == 4 ? 276 : 412;
  uint32_t part[kStage16][kPartToken];
  float kf[kStage16][kKfToken];
  float v[kStage16][LM::kWaves * LM::kCols];
};

template <class Tag, int Layout>
struct alignas(16) Scan16Lds {
  Stage16<Tag, Layout> st[2];
  // Token t's alpha, beta, alpha / kScale and k_hat . q_hat at [t / 64 % 2][t % 64].
  float gate[2][kGateTokens][4];
};

// A lane's share of four tokens of a stage (a round): 16-lane row r = lane / 16
// holds token 4 u + r of round u, lane x = lane % 16 of it elements 8 x .. 8 x + 7
// of its q and k and a sixteenth of its v.
static_assert(kStage16 == 4 * 4, "four rounds of four tokens");

template <int Layout>
struct Round16 {
  static constexpr int kV = Scan16Map<Layout>::kWaves * Scan16Map<Layout>::kCols / 16;
  float q[8], k[8], v[kV];
};

struct Scan16Row {
  const float *q, *k, *v;  // the row's first token
  size_t qk_tok, v_tok;    // token strides
};

template <int N>
__device__ __forceinline__ void load16(const float* p, float (&out)[N]) {
  if constexpr (N == 8) {
    float lo[4], hi[4];
    loadN<4>(p, lo);
    loadN<4>(p + 4, hi);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = lo[i], out[4 + i] = hi[i];
  } else {
    loadN<N>(p, out);
  }
}

// Round u of the stage at token t0; the row has len tokens.
template <int Layout>
__device__ __forceinline__ void load_round16(Round16<Layout>& r, int lane, const Scan16Row& in,
                                             int t0, int u, int len) {
  const int t = t0 + 4 * u + (lane >> 4), x = lane & 15;
  if (t < len) {
    load16<8>(in.q + (size_t)t * in.qk_tok + 8 * x, r.q);
    load16<8>(in.k + (size_t)t * in.qk_tok + 8 * x, r.k);
    constexpr int kV = Round16<Layout>::kV;
    load16<kV>(in.v + (size_t)t * in.v_tok + kV * x, r.v);
  }
}

// Sum over a vector held as eight consecutive elements by the lanes of a
// 16-lane row, from the lane's four pair sums: the wave butterfly's tree
// (gdn_tile.h, wave_sum over pairs), so the decode's bits.
__device__ __forceinline__ float row_tree(float p0, float p1, float p2, float p3) {
  return add_xor8(add_xor4(add_xor2(add_xor1((p0 + p1) + (p2 + p3)))));
}
__device__ __forceinline__ float row_dot(const float (&a)[8], const float (&b)[8]) {
  return row_tree(a[0] * b[0] + a[1] * b[1], a[2] * b[2] + a[3] * b[3], a[4] * b[4] + a[5] * b[5],
                  a[6] * b[6] + a[7] * b[7]);
}

// One vector's parts into a stage token.
template <class Tag>
__device__ __forceinline__ void write_parts(const float (&x)[8], uint32_t* dst) {
#pragma unroll
  for (int g = 0; g < kRowGroups; ++g) {
    uint32_t p[Parts<Tag>::kSplit];
    Parts<Tag>::split2(x[g], x[g + 4], p);  // rows i0 and i0 + 1 of row group g
#pragma unroll
    for (int s = 0; s < Parts<Tag>::kSplit; ++s) dst[s * kPartRow + g * 4] = p[s];
  }
}

template <class Tag, int Layout>
__device__ __forceinline__ void write_round16(const Round16<Layout>& r, int lane, int u,
                                              Stage16<Tag, Layout>& st, float (*gate)[4]) {
  const int tok = 4 * u + (lane >> 4), x = lane & 15;
  float q[8], k[8];
  constexpr float kScale = Parts<Tag>::kScale, kInv = 1.f / kScale;
  const float qi = rsqrtf(row_dot(r.q, r.q) + kL2Eps) * kScale;
  const float ki = rsqrtf(row_dot(r.k, r.k) + kL2Eps) * kScale;
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = r.q[i] * qi, k[i] = r.k[i] * ki;
  const float kq = row_dot(k, q) * (kInv * kInv);
  // Rows 8 x + kk: block x / 4, row group kk % 4, index 2 (x % 4) + kk / 4.
  const int w = x >> 2, x4 = x & 3;
  uint32_t* part = &st.part[tok][w * 16 + x4];
  write_parts<Tag>(k, part);
  write_parts<Tag>(q, part + Parts<Tag>::kQ * kPartRow);
  float* kf = &st.kf[tok][(w >> 1) * kKfHalf + 8 * (x4 & 1) + 2 * (w & 1) + (x4 >> 1)];
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) kf[16 * (kk & 3) + 4 * (kk >> 2)] = k[kk] * kInv;
  constexpr int kV = Round16<Layout>::kV;
  float* vd = &st.v[tok][kV * x];
  if constexpr (kV == 8) {
    const float lo[4] = {r.v[0], r.v[1], r.v[2], r.v[3]};
    const float hi[4] = {r.v[4], r.v[5], r.v[6], r.v[7]};
    storeN<4>(vd, lo);
    storeN<4>(vd + 4, hi);
  } else {
    storeN<kV>(vd, r.v);
  }
  if (x == 0) gate[tok][3] = kq;
}

template <class Tag, class Gates>
__device__ __forceinline__ void write_gate16(const Gates& gates, const GateRaw& r,
                                             const GateConst& gc, float (&dst)[4]) {
  const float alpha = gates.alpha_of(r, gc);
  dst[0] = alpha;
  dst[1] = gates.eval_beta(r);
  dst[2] = alpha * (1.f / Parts<Tag>::kScale);
}

// A token's operands of the state products (one per block the lane holds),
// and of the update and the readout.
template <class Tag, int Layout>
struct Tok16A {
  u32x4 a[Scan16Map<Layout>::kNB][Parts<Tag>::kFrags];
};
template <int Layout>
struct Tok16B {
  float kf[2 * Scan16Map<Layout>::kNB];
  float v;
  float alpha, beta, alpha_s, kq;
};

template <class Tag, int Layout>
__device__ __forceinline__ void read_a(const Stage16<Tag, Layout>& st, int tok,
                                       const Scan16Map<Layout>& L, int s,
                                       Tok16A<Tag, Layout>& t) {
#pragma unroll
  for (int f = 0; f < Parts<Tag>::kFrags; ++f)
    t.a[s][f] = *reinterpret_cast<const u32x4*>(
        &st.part[tok][Parts<Tag>::part_of(f, L.j) * kPartRow +
                      16 * (Scan16Map<Layout>::block_of(0, L.j) + s) + 4 * L.g]);
}

template <class Tag, int Layout>
__device__ __forceinline__ void read_b(const Stage16<Tag, Layout>& st, const float (*gate)[4],
                                       int tok, const Scan16Map<Layout>& L, Tok16B<Layout>& t) {
  constexpr int NB = Scan16Map<Layout>::kNB;
  float gt[4];
  loadN<4>(gate[tok], gt);
  t.alpha = gt[0], t.beta = gt[1], t.alpha_s = gt[2], t.kq = gt[3];
  t.v = st.v[tok][L.col];
  const float* p = &st.kf[tok][(4 * L.g + (L.j & 3)) * 4];
  if constexpr (NB == 4) {
    float lo[4], hi[4];
    loadN<4>(p, lo);
    loadN<4>(p + kKfHalf, hi);
#pragma unroll
    for (int i = 0; i < 4; ++i) t.kf[i] = lo[i], t.kf[4 + i] = hi[i];
  } else if constexpr (NB == 2) {
    loadN<4>(p + L.h * kKfHalf, t.kf);
  } else {
    loadN<2>(p + (L.h >> 1) * kKfHalf + 2 * (L.h & 1), t.kf);
  }
}

// The lane's state: p[s][m] = rows i = 2 m (low half) and 2 m + 1 of block s
// of its column.
template <class Tag, int Layout>
struct State16 {
  static constexpr int NB = Scan16Map<Layout>::kNB;
  u32x4 p[NB];
  __device__ __forceinline__ void load(const Scan16Map<Layout>& L, const uint16_t* tile) {
#pragma unroll
    for (int s = 0; s < NB; ++s)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const uint16_t* a = tile + L.row(s, 2 * m) * kHD + L.col;
        p[s][m] = (uint32_t)__builtin_nontemporal_load(a) |
                  ((uint32_t)__builtin_nontemporal_load(a + kRowGroups * kHD) << 16);
      }
  }
  __device__ __forceinline__ void store(const Scan16Map<Layout>& L, uint16_t* tile) const {
#pragma unroll
    for (int s = 0; s < NB; ++s)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        uint16_t* a = tile + L.row(s, 2 * m) * kHD + L.col;
        __builtin_nontemporal_store((uint16_t)p[s][m], a);
        __builtin_nontemporal_store((uint16_t)(p[s][m] >> 16), a + kRowGroups * kHD);
      }
  }
};

// The state products of one token, d[s] of the lane's block s.
template <class Tag, int Layout>
struct Prod16 {
  f32x4v d[Scan16Map<Layout>::kNB][Parts<Tag>::kFrags];
};

template <class Tag, int Layout>
__device__ __forceinline__ void products16(const Tok16A<Tag, Layout>& t,
                                           const State16<Tag, Layout>& S, int s,
                                           Prod16<Tag, Layout>& out) {
#pragma unroll
  for (int f = 0; f < Parts<Tag>::kFrags; ++f) out.d[s][f] = Parts<Tag>::mfma(t.a[s][f], S.p[s]);
}

// The column total of the blocks' sums, as (t0 + t1) + (t2 + t3). t: the
// lane's blocks' sums, added up in that order. Where a column is split over
// lanes, only the lanes whose group stands for their own h hold its sum: the
// others put in -0, which adds nothing, and the exchange over the lane groups
// (xor 16, 32) leaves the sum in all of them; then the h are added (xor 4, 8).
template <int Layout>
__device__ __forceinline__ float column_total16(const Scan16Map<Layout>& L, float t) {
  constexpr int NB = Scan16Map<Layout>::kNB;
  if constexpr (NB == 4) {
    return t;
  } else if constexpr (NB == 2) {
    return add_xor8(add_xor16((L.g & 1) == L.h ? t : -0.f));
  } else {
    return add_xor8(add_xor4(add_xor32(add_xor16(L.g == L.h ? t : -0.f))));
  }
}
template <int NB>
__device__ __forceinline__ float block_sum16(const float (&t)[NB]) {
  if constexpr (NB == 4) return (t[0] + t[1]) + (t[2] + t[3]);
  else if constexpr (NB == 2) return t[0] + t[1];
  else return t[0];
}

// Blocks whose operands are read before a token's update begins; the others'
// reads follow block by block. All of them where the registers allow; bf16's
// operands are twice the registers, and all of them at once would spill under
// the 168 that twelve-wave workgroups leave (layout 2, and layout 1 in the
// planned kernel, kTight: 0.38 us a token instead of 0.36 with all of them).
template <class Tag, int Layout, bool kTight>
constexpr int kAhead16 = Parts<Tag>::kFrags == 1 ? 4 : (Layout == 2 ? 1 : (kTight ? 2 : 4));

// One token: from its products D (and its operands b), the update of the
// state, with the next token's products (operands an) issued block by block
// behind it, into D. neg_zero: four -0 registers, the accumulator that makes
// the outer-product MFMA an exact rounded product (adding -0 changes nothing).
template <class Tag, int Layout, bool kTight>
__device__ __forceinline__ float token16(const Scan16Map<Layout>& L, State16<Tag, Layout>& S,
                                         Prod16<Tag, Layout>& D, Tok16A<Tag, Layout>& an,
                                         const Stage16<Tag, Layout>& st, int next,
                                         const Tok16B<Layout>& b, f32x4v neg_zero) {
  using P = Parts<Tag>;
  constexpr int NB = Scan16Map<Layout>::kNB;
  float tk[NB], tq[NB];
#pragma unroll
  for (int s = 0; s < NB; ++s) tk[s] = P::kv(D.d[s]);
  const float kv = column_total16<Layout>(L, block_sum16<NB>(tk));
  const float delta = delta_of(b.v, b.alpha_s, b.beta, kv);
  // k_hat * delta for the lane's rows: the 4x4x1 MFMA's block (lane / 4) takes
  // four rows of the lane's row group and block, one per lane of the quad, and
  // four columns' delta; each lane gets its column's four rows. Issued back to
  // back: a switch between VALU and MFMA costs about 7 clocks each time
  // (config 2's eight rows at T = 384 in layout 1 0.549 -> 0.501 us a token).
  f32x4v x[NB][2];
#pragma unroll
  for (int s = 0; s < NB; ++s)
#pragma unroll
    for (int u = 0; u < 2; ++u)
      x[s][u] = __builtin_amdgcn_mfma_f32_4x4x1f32(b.kf[2 * s + u], delta, neg_zero, 0, 0, 0);
#pragma unroll
  for (int s = 0; s < NB; ++s) tq[s] = P::sq(D.d[s]);
  const float sqb = block_sum16<NB>(tq);
  // bf16 state has no mixed-precision fma: in layout 8, whose one wave per SIMD
  // waits for delta's chain here, it is widened meanwhile (0.205 -> 0.193 us a
  // token; layout 4, with twice the elements, is slower so, 0.237 -> 0.245).
  constexpr bool kWide = std::is_same<Tag, BF16>::value && NB == 1;
  float wide[kWide ? NB : 1][8];
  if constexpr (kWide) {
#pragma unroll
    for (int s = 0; s < NB; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) wide[s][i] = half_of<Tag>(S.p[s][i >> 1], i & 1);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < NB; ++s) {
    if (s + kAhead16<Tag, Layout, kTight> < NB) read_a<Tag, Layout>(st, next, L, s + kAhead16<Tag, Layout, kTight>, an);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      float s0, s1;
      if constexpr (kWide) {
        s0 = wide[s][2 * m];
        s1 = wide[s][2 * m + 1];
      } else {
        s0 = half_of<Tag>(S.p[s][m], 0);
        s1 = half_of<Tag>(S.p[s][m], 1);
      }
      const float n0 = opaque(fmaf(b.alpha, s0, x[s][m >> 1][2 * (m & 1)]));
      const float n1 = opaque(fmaf(b.alpha, s1, x[s][m >> 1][2 * (m & 1) + 1]));
      S.p[s][m] = pack_pair<Tag>(n0, n1);
    }
    products16<Tag, Layout>(an, S, s, D);
  }
  const float sq = column_total16<Layout>(L, sqb);
  return readout_of(b.alpha_s, sq, delta, b.kq);
}

// The live tokens of one row's tile columns (a workgroup's share): kWaves waves
// run the tokens and kPrep prepare the stages. A token wave's issue slots are
// what the scan is short of, and a stage's preparation (norms, parts, gates) is
// a long chain with many waits; on waves of its own it runs beside the tokens,
// one stage ahead, and meets them at one barrier a stage.
// y's element from its fp32 value: as it is, or rounded to bf16 (the readout's
// first step, for callers that would do it next).
__device__ __forceinline__ void put_y(float* p, float y) { *p = y; }
__device__ __forceinline__ void put_y(uint16_t* p, float y) { *p = (uint16_t)pack_bf16x2(y, 0.f); }

template <class Tag, class Gates, class YT, int Layout, bool kTight = false>
__device__ __forceinline__ void prefill_tile16(uint16_t* __restrict__ pool,
                                               const int* __restrict__ slot_idx,
                                               const float* __restrict__ q,
                                               const float* __restrict__ k,
                                               const float* __restrict__ v, const Gates& gates,
                                               YT* __restrict__ y, int H,
                                               int heads_per_group, int T, long qk_tok, long v_tok,
                                               int b, int h, int part, int len,
                                               Scan16Lds<Tag, Layout>& lds) {
  using LM = Scan16Map<Layout>;
  using St = Stage16<Tag, Layout>;
  constexpr int kWgCols = LM::kWaves * LM::kCols;
  constexpr int kGateStages = kGateTokens / kStage16;
  const int g = h / heads_per_group;
  const int c0 = part * kWgCols;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // A layout's waves beyond kThreads (the planned kernel launches the most any
  // layout needs) end here; the workgroup's barriers count the live ones.
  if (wave >= LM::kWaves + LM::kPrep) return;
  const Scan16Row in{q + (size_t)b * T * qk_tok + (size_t)g * kSS,
                     k + (size_t)b * T * qk_tok + (size_t)g * kSS,
                     v + (size_t)b * T * v_tok + (size_t)h * kHD + c0, (size_t)qk_tok,
                     (size_t)v_tok};
  auto gate_slot = [&](int s) {
    return &lds.gate[(s / kGateStages) & 1][(s % kGateStages) * kStage16];
  };

  if (wave >= LM::kWaves) {
    const int u = wave - LM::kWaves;
    __builtin_amdgcn_s_setprio(1);
    const GateConst gc = gates.tile_consts(h);
    auto write_gates = [&](int t0) {  // of tokens t0 .. t0 + 63
      const int t = t0 + lane;
      if (t < len)
        write_gate16<Tag>(gates, gates.load_live(b, h, t, H, T), gc,
                          lds.gate[(t0 / kGateTokens) & 1][lane]);
    };
    Round16<Layout> r;
    load_round16<Layout>(r, lane, in, kStage16, u, len);
    if (u == 0) write_gates(0);
    __syncthreads();
    int stage = 0;
    for (int t0 = 0; t0 < len; t0 += kStage16, ++stage) {
      // The next stage, into the buffer that every wave left behind at the
      // last barrier, and the loads of the one after it; tokens past the row's
      // end write what no token reads.
      if (t0 + kStage16 < len) {
        write_round16<Tag, Layout>(r, lane, u, lds.st[(stage + 1) & 1], gate_slot(stage + 1));
        load_round16<Layout>(r, lane, in, t0 + 2 * kStage16, u, len);
      }
      // Gates of the next 64 tokens, at the start of these 64.
      if (stage % kGateStages == 0 && u == ((stage / kGateStages) & 3))
        write_gates(t0 + kGateTokens);
      __syncthreads();
    }
  } else {
    const LM L(threadIdx.x);
    const int slot = slot_idx[b];
    uint16_t* tile = pool + ((size_t)slot * H + h) * (kSS * kHD) + c0;
    State16<Tag, Layout> S;
    S.load(L, tile);
    // The first stage, a round a wave.
    if (wave < 4) {
      Round16<Layout> r;
      load_round16<Layout>(r, lane, in, 0, wave, len);
      write_round16<Tag, Layout>(r, lane, wave, lds.st[0], lds.gate[0]);
    }
    __syncthreads();

    f32x4v neg_zero = {-0.f, -0.f, -0.f, -0.f};
    asm("" : "+v"(neg_zero));
    const size_t y_tok = (size_t)H * kHD;
    // Where the lane's y goes: its slot's token of each kSlots tokens.
    YT* yp = y + (((size_t)b * T + L.slot) * H + h) * kHD + c0 + L.col;
    float yv = 0.f;
    int stage = 0;
    for (int t0 = 0; t0 < len; t0 += kStage16, ++stage) {
      const int n = min(kStage16, len - t0);
      const St& st = lds.st[stage & 1];
      const float(*gate)[4] = gate_slot(stage);
      Tok16A<Tag, Layout> a;
      Tok16B<Layout> bb[2];
      Prod16<Tag, Layout> D;
      read_b<Tag, Layout>(st, gate, 0, L, bb[0]);
#pragma unroll
      for (int s = 0; s < LM::kNB; ++s) {
        read_a<Tag, Layout>(st, 0, L, s, a);
        products16<Tag, Layout>(a, S, s, D);
      }
      // Token j, its operands in bb[i]; the next token's are read meanwhile.
      // Reads past the stage's live tokens stay inside it and go unused.
      auto step = [&](int j, int i) {
        const int jn = min(j + 1, kStage16 - 1);
#pragma unroll
        for (int s = 0; s < LM::kNB && s < kAhead16<Tag, Layout, kTight>; ++s) read_a<Tag, Layout>(st, jn, L, s, a);
        read_b<Tag, Layout>(st, gate, jn, L, bb[i ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
        const float yy = token16<Tag, Layout, kTight>(L, S, D, a, st, jn, bb[i], neg_zero);
        yv = L.slot == (j & (LM::kSlots - 1)) ? yy : yv;
      };
      int j = 0;
      for (; j + 4 <= n; j += 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) step(j + i, i & 1);
        if (((j + 4) & (LM::kSlots - 1)) == 0) {
          put_y(yp, yv);
          yp += LM::kSlots * y_tok;
        }
      }
      if (j < n) {  // the row's last tokens
        step(j, 0);
        if (j + 1 < n) step(j + 1, 1);
        if (j + 2 < n) step(j + 2, 0);
      }
      __syncthreads();
    }
    const int rest = len & (LM::kSlots - 1);
    if (L.slot < rest) put_y(yp, yv);
    S.store(L, tile);
  }

  // Zeros at the pad positions, the workgroup's columns, 16 bytes per thread.
  constexpr int kPer = 16 / sizeof(YT), kV = kWgCols / kPer;
  for (int e = threadIdx.x; e < (T - len) * kV; e += LM::kThreads) {
    const int t = len + e / kV, c = c0 + kPer * (e % kV);
    __builtin_nontemporal_store((u32x4){0u, 0u, 0u, 0u},
                                reinterpret_cast<u32x4*>(y + (((size_t)b * T + t) * H + h) * kHD + c));
  }
}

}  // namespace braid
