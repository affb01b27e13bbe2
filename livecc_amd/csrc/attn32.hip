// LLM prefill attention, second generation: 32-row query tiles on the 32x32x16 bf16 MFMA, K/V tiles shared by the G query heads of
// one KV head through an LDS-DMA ring.  Replaces HF modeling_qwen2_vl.py:537-556 (Qwen2VLAttention core: causal, bottom-right aligned,
// GQA) for prefill rows, same contract as attn_shared_kernel<128, NQ, 1, G> in attention.hip (which stays as variant 2).
//
// Why (profiles/r03/pmc_attn_summary.json, 8 streams x 386 rows x 6k keys on attn_shared_kernel<128,1,1,7>): 25 % MFMA busy, 8.3 VALU
// instructions per MFMA, 16 ds_read_b128 per 16 MFMAs of 16 cycles each -- per CU and 32-key tile the LDS reads (112 KB / 256 B/clk
// = 437 clk), the MFMAs (448 clk) and the softmax VALU work cost about the same and only partly overlap: 0.54 PF.  One wave now owns
// 32 query rows of one head:
//   * S^T[32 keys][32 queries] = K . Q^T  is 8 MFMAs of 32 cycles (k = 16 each), O^T[128 d][32 queries] += V^T . P^T another 8: the
//     same 16 ds_read_b128 per tile now feed 512 MFMA cycles instead of 256 -- LDS traffic per flop halves;
//   * in the 32x32 C/D layout a lane owns ONE query column (l & 31) and 16 keys, so the row maximum / sum are 15 in-lane steps + ONE
//     cross-lane step (xor 32) instead of 7 + 2 per 8 scores;
//   * the K rows of a tile are fetched in a permuted order (bits 2 and 3 of the row index swapped), so that the 16 scores a lane
//     ends up with are exactly the 2 x 8 consecutive keys its B-operand slots of the two P.V MFMAs need: P goes from the softmax
//     registers into the MFMA with 8 v_cvt_pk and no cross-lane traffic at all.
// Layouts (gfx950 v_mfma_f32_32x32x16_bf16): A lane l = A[i = l & 31][k = (l >> 5) * 8 + e]; B lane l = B[k = (l >> 5) * 8 + e][j = l & 31];
// C/D lane l, r = 0..15: D[i = 8 * (r >> 2) + 4 * (l >> 5) + (r & 3)][j = l & 31].
// With key(i) = tile * 32 + swap23(i): score register r of lane-half hh holds key offset 16 * (r >> 3) + 8 * hh + (r & 7).
#include <cstdlib>
#include <type_traits>

#include <algorithm>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace lcc {

typedef __attribute__((ext_vector_type(16))) float f32x16;

LCC_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
LCC_DEVICE int swap23(int i) { return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1); }
LCC_DEVICE float vmax(float a, float b) { return __builtin_fmaxf(a, b); }
LCC_DEVICE float vmax3(float a, float b, float c) { return __builtin_fmaxf(__builtin_fmaxf(a, b), c); }   // hipcc emits v_max3_f32
// max over the two lanes l and l ^ 32 with ONE v_permlane32_swap (instead of a ds_bpermute round trip through the LDS crossbar)
LCC_DEVICE float xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
LCC_DEVICE float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <class F, int... I>
LCC_DEVICE void unrolled_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
LCC_DEVICE void unrolled(F&& f) { unrolled_of(f, std::make_integer_sequence<int, N>{}); }      // f(0) .. f(N - 1), the index a constant

// ------------------------------------------------------------------------------------------------------------------------------
// The key loop shared by the LLM prefill kernel (D = 128), the causal multi-head kernel and the ViT kernel (D = 80): software pipeline, a pair of key
// tiles an iteration.  The softmax of pair P (vector pipe) is issued next to the MFMAs that do not depend on it -- the P . V of pair P - 1 and the K . Q^T of
// pair P + 1 (matrix pipe: 32 x 32 cycles at D = 128) -- in ONE basic block: every fragment read FRAG_LEAD MFMAs ahead of its use, the vector work dealt out in
// steps (Attn32Steps), the DMA pieces of pair P + 2 spread between them: a wave always has matrix AND vector work in flight.
//
// Ring of three pair-stages.  Slot t holds what the iteration of tile t multiplies -- K of tile t + 2 and V^T of tile t - 2 -- so a pair needs its own two slots
// only: at the top of the iteration of pair (t, t + 1) its slots have landed (counted vmcnt: only the next pair's, issued one iteration ago, may still
// be in flight; barrier: every wave's pieces) and the slots of the pair before receive pair t + 4.  The iteration enters with the scores of tiles t and t + 1 and leaves with
// those of t + 2 and t + 3.
//
// Reference of the softmax: the row's running maximum, that of the pair included.  All scores of the pair are there when the iteration begins, so every
// probability is at most one, the row's largest IS one and no rounding touches it.  O, which is one pair behind, is brought to the maximum by the factor alpha at
// the top of the next iteration, if any row of the wave needs it.
//   * A reference that moves rarely (a first tile's maximum plus whole powers of two: no rescale in most iterations) was taken back: the row's largest probability is
//     then rounded to bf16 like any other.  Error against 64 bits (2-norm, 1e-3), 386 rows on 386 keys / 64 on 8,000 with a bias, normal keys and values of 1 / 2 / 4:
//     2.02 / 2.09 / 2.14 and 2.34 / 2.34 / 2.34 there, 1.96 / 1.82 / 1.72 and 1.89 / 1.80 / 1.72 here (a maximum per tile: 1.94 / 1.81 / 1.72 and 1.89 / 1.79 / 1.71).
//   * Scores of one tile alone at the top (the second tile's maximum a region later): two places to rescale O, and a branch in each.
//   * Each row decides by its own scores (both lanes of its column), so its bits do not depend on its neighbours in the wave.
// Measured (us; one region of 16 / 11 MFMAs a tile with fragment-order gathers -> rare moves -> here): 4,096 rows on 8k keys 667 -> 589 -> 598 (1.01 PF), 386 rows
// on 2k keys in five splits 38.1 -> 34.2 -> 34.9, 8 x 386 rows on 1.1k 102 -> 84.0 -> 87.0; with a bias, 4,096 rows on 4k 577 -> 516 -> 420; tower, 18 slices of 880
// patches 174 -> 117 -> 122, one of 1,456 32.8 -> 29.4 -> 30.0.  What bounds it: the vector pipe beside the matrix pipe.
//
// LDS image of a slot: rows as they lie in memory, so that a DMA instruction copies whole runs of lines (K: 32 keys x 2 D bytes; V^T: DV rows x 64 bytes)
// instead of 64 separate 16-byte chunks, each a line of its own for the address path (a 4-wave block of the tower kernel spent 15 of its 42 us on that).  A row's
// 16-byte chunks are permuted (kx, vx) so that the fragment reads -- one chunk of 16 rows at a time -- touch every bank once; K rows of 256 bytes
// also shift by a chunk every four rows (their DMA instruction).
//   mlim: tiles reaching past it need the mask (causal diagonal / end of the key range); lim: this lane's effective key limit.
//
// Fragments are read four MFMAs ahead, at 128 channels five, as many as there are registers for: 4,096 rows on 8k keys 631 -> 626 us, 8 x 386 on 1.1k 90.6 -> 88.9,
// 1,131 rows 36.2 -> 35.3; six 629, 89.0 and 35.3, three 638, 90.2 and 36.0.  At 80 channels five and six are no faster (18 slices of 880 123 / 124 / 127).
// Measured and not taken: the two waves of a SIMD in opposite phases (matrix work of one beside the softmax of the other): 11 % slower than the
// instruction-by-instruction interleave; all fragments of a region read a region ahead: 64 registers, spills.
// LM (the tower kernel): the softmax denominator comes out of the P . V MFMAs -- the V^T rows 80..95 of the third d-tile do not exist at d = 80 and
// are ONES, so O^T rows 80..95 accumulate sum_k bf16(P) under the same rescale as O -- instead of 16 additions per region.  l then sums the ROUNDED
// probabilities the numerator uses (fp32 accumulation either way).
// D = channels of q / k, DV = channels of v.  BIAS: slope (pos - key) is taken off the scaled scores (slope in units of log2), pos = this lane's query:
// K.Q^T is added to it instead of to zero.
struct Kv32 {                   // keys and values of one (stream, head); all wave-uniform
  const bf16_t *k, *v;          // tile 0
  unsigned k_row, v_row;        // bytes between keys of K, between channels of V^T
  size_t k_tile, v_tile;        // bytes between 32-key tiles
  int ntile, nkeys;             // tiles; CLAMP: keys that exist (the last tile's rows beyond them are not read)
};
template <int D, int DV>
struct Attn32Image {
  static constexpr int CR = D / 8, DT = (DV + 31) / 32, KPD = D / 16, VPD = DV / 16, NPD = KPD + VPD;      // chunks of a K row; DMA instructions of K, V
  static constexpr int KB = D == 128 ? 8 * 1040 : 64 * D, VB = DT * 2048, SLOT = KB + VB, BYTES = 6 * SLOT;
  LCC_DEVICE static int kx(int row) { return D == 128 ? (row & 3) * 4 : D == 64 ? (row >> 1) & 7 : (row >> 3) & 1; }
  LCC_DEVICE static int vx(int d) { return (d >> 2) & 3; }
};

// The 32 probabilities of a pair are formed two at a time beside its MFMAs: how many twos up to behind MFMA i (17: the last one summed, too).  Evenly, or with
// wide values (whose P.V leaves the time) each tile's before the MFMAs that overwrite its scores: the new scores then take the old ones' registers.
template <int VP, int KP>
struct Attn32Steps {
  static constexpr int formed(int i) {
    constexpr int N = 2 * (VP + KP), A = 2 * VP - 1, B = 2 * VP + KP - 1;
    if (i < 5) return 0;
    if (VP < 8) return i == N - 1 ? 17 : (i - 4) * 16 / (N - 6);
    if (i < A) return (i - 4) * 8 / (A - 5);
    return i >= B ? 17 : i == B - 1 ? 16 : 8 + (i - A + 1) * 8 / (B - A);
  }
};
template <int D, int DV, int NWAVE, bool LM, bool BIAS = false, bool CLAMP = false>
LCC_DEVICE void attn32_key_loop(unsigned char* alds, const Kv32& kv, const u32x4 (&qf)[D / 16], int tb, int te, int mlim, int lim, float scale_log2e,
                                bool active, int lane, int wave, int hh, f32x16 (&o)[(DV + 31) / 32], float& m_run, float& l_run, float slope = 0.f, int pos = 0) {
  using Im = Attn32Image<D, DV>;
  constexpr int KP = D / 16, DT = Im::DT, VP = 2 * DT, NP = KP + VP, FRAG_LEAD = D == 128 ? 5 : 4;
  using Steps = Attn32Steps<VP, KP>;
  constexpr int NPD = Im::NPD, PWP = (2 * NPD + NWAVE - 1) / NWAVE, PK = (Im::KPD + NWAVE - 1) / NWAVE;     // DMA pieces of a wave: a pair; K of one tile
  m_run = -INFINITY;
  if (te <= tb) return;                                 // (block-uniform: a key split without a tile)
  const unsigned lds0 = lds_addr(alds);
  const float bias_raw = BIAS ? slope / scale_log2e : 0.f;
  const int col = lane & 31;

  // DMA: this wave's pieces of a pair.  Surplus slots copy the last piece again (same bytes, same place).  What a piece needs in every pair -- its operand, tiles from the
  // pair's, row bytes and place in a slot -- is kept in scalar registers: formed anew, a pair of the four-wave tower kernel had 101 scalar instructions
  // beside 202 others, now 68 (eight waves 60 / 42, LLM prefill 63 / 45); one chunk's tower 4,079 / 4,042 us in turn on one card, eight chunks' the same
  struct Piece { const char* base; unsigned stride, row, at; int dt, lo; };
  Piece pc[PWP];
  unsigned off[PWP], prow[CLAMP ? PWP : 1];
#pragma unroll
  for (int j = 0; j < PWP; ++j) {
    const int u = min(j * NWAVE + wave, 2 * NPD - 1), r = u >= NPD ? 1 : 0, p = u - r * NPD;
    const bool is_k = p < Im::KPD;
    pc[j].base = is_k ? reinterpret_cast<const char*>(kv.k) : reinterpret_cast<const char*>(kv.v);
    pc[j].stride = (unsigned)(is_k ? kv.k_tile : kv.v_tile);
    pc[j].row = is_k ? kv.k_row : 0u;
    pc[j].at = (unsigned)(r * Im::SLOT + (is_k ? p * (D == 128 ? 1040 : 1024) : Im::KB + (p - Im::KPD) * 1024));
    pc[j].dt = is_k ? r + 2 : r - 2;
    pc[j].lo = is_k ? 0 : tb;
    if (p < Im::KPD) {
      const int row = (p * 64 + lane) / Im::CR, c = (p * 64 + lane) % Im::CR;
      off[j] = (CLAMP ? 0u : (unsigned)row * kv.k_row) + (unsigned)((c ^ Im::kx(row)) * 16);
      if (CLAMP) prow[j] = row;
    } else {
      const int d = (p - Im::KPD) * 16 + (lane >> 2);
      off[j] = (unsigned)d * kv.v_row + (unsigned)(((lane & 3) ^ Im::vx(d)) * 16);
      if (CLAMP) prow[j] = 0u;
    }
  }
  auto piece = [&](const char* base, unsigned stride, int tile, unsigned row_bytes, unsigned o_lane, unsigned row, unsigned at) {      // tile: in range
    if (CLAMP) o_lane += __umul24(min(row, (unsigned)(kv.nkeys - 1 - tile * 32)), row_bytes);      // no branch: this is inside the pair's basic block
    glds16_base(base + (unsigned long long)stride * (unsigned)tile, o_lane, at);
  };
  auto issue = [&](int j, int t, int ps) {              // piece j of the pair (t, t + 1) into pair-stage ps
    const int tile = min(max(t + pc[j].dt, pc[j].lo), kv.ntile - 1);
    piece(pc[j].base, pc[j].stride, tile, pc[j].row, off[j], CLAMP ? prow[CLAMP ? j : 0] : 0u, lds0 + (unsigned)(2 * ps * Im::SLOT) + pc[j].at);
  };
  // fragment addresses inside a slot: K row swap23(col), chunk 2 ks + hh; V^T row 32 dt + col, chunk 2 s + hh
  constexpr int NKA = D == 80 ? 1 : 4;
  int ka[NKA], va[2];
  {
    const int row = swap23(col), r0 = D == 128 ? (row >> 2) * 1040 + (row & 3) * 256 : row * D * 2, x = Im::kx(row);
#pragma unroll
    for (int i = 0; i < NKA; ++i) ka[i] = r0 + (((D == 128 ? 4 * i + hh : 2 * i + hh) ^ x) * 16);
#pragma unroll
    for (int s = 0; s < 2; ++s) va[s] = Im::KB + col * 64 + (((2 * s + hh) ^ Im::vx(col)) * 16);
  }
  auto kfrag = [&](const unsigned char* slot, int ks) {
    return *reinterpret_cast<const u32x4*>(slot + ka[D == 128 ? ks >> 1 : D == 80 ? 0 : ks] + (D == 128 ? (ks & 1) * 32 : D == 80 ? ks * 32 : 0));
  };
  auto vfrag = [&](const unsigned char* slot, int i) { return *reinterpret_cast<const u32x4*>(slot + va[i & 1] + (i >> 1) * 2048); };

  auto clear = [&](int t, f32x16& sc) {                           // what K.Q^T of tile t is added to: the bias, in units of unscaled scores
    // the distance as a whole number, so that near keys keep theirs at any position (slope times position, cancelled against slope times key, is off by
    // up to 8e-3 in log2 units at 131,000)
    const float base = BIAS ? bias_raw * (float)(t * 32 + 8 * hh - pos) : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = BIAS ? fmaf(bias_raw, (float)(16 * (r >> 3) + (r & 7)), base) : 0.f;
  };
  bf16x8 p_prev[4];                                     // P of the previous pair, its P . V still pending
#pragma unroll
  for (int i = 0; i < 4; ++i) p_prev[i] = as_bf16x8((u32x4){0u, 0u, 0u, 0u});
  f32x16 sc[2];
  float alpha = 1.f;                                    // what brings O (pairs before the previous one) to the maximum that p_prev was taken against
  int st = 0;                                           // pair-stage of the pair
  // one pair: softmax of tiles t and t + 1 (vector pipe) beside P.V of t - 2 and t - 1, K.Q^T of t + 2 and t + 3 (matrix pipe)
  auto pair = [&](auto masked_tag, int t) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    // the two copies of the pair keep their fragment reads: shared, they would all sit in front of the branch between them
    if (MASKED) asm volatile("; masked pair" ::: "memory"); else asm volatile("; whole pair" ::: "memory");
    const unsigned char* slot[2] = {alds + 2 * st * Im::SLOT, alds + (2 * st + 1) * Im::SLOT};
    const int ps = st == 0 ? 2 : st - 1;
    u32x4 f[FRAG_LEAD + 1];
    auto read = [&](int i) { return i < 2 * VP ? vfrag(slot[i / VP], i % VP) : kfrag(slot[(i - 2 * VP) / KP], (i - 2 * VP) % KP); };
#pragma unroll
    for (int i = 0; i < FRAG_LEAD; ++i) f[i] = read(i);
    // the vector work in steps: the maximum of eight scores (four of them), the new reference, then two probabilities at a time
    f32x16 x[2] = {sc[0], sc[1]};
    float mx[2] = {-INFINITY, -INFINITY}, psum[2] = {0.f, 0.f}, m_use = 0.f, al = 1.f;
    u32x4 w[4];
    auto settle = [&](auto kc) {              // they are there by now: without this the compiler moves pure arithmetic behind the MFMAs, in front of its use
      constexpr int r = decltype(kc)::value >> 3, e = (decltype(kc)::value & 7) * 2;
      float a = x[r][e], b = x[r][e + 1];
      if constexpr (LM) asm volatile("" : "+v"(a), "+v"(b));
      else {
        psum[0] += a; psum[1] += b;           // the denominator sums the probabilities unrounded
        asm volatile("" : "+v"(a), "+v"(b), "+v"(psum[0]), "+v"(psum[1]));
      }
      x[r][e] = a; x[r][e + 1] = b;
    };
    auto step = [&](auto nc) {
      constexpr int n = decltype(nc)::value;
      if constexpr (n < 4) {
        constexpr int r = n >> 1, e0 = (n & 1) * 8;
#pragma unroll
        for (int e = e0; e < e0 + 8; ++e)
          if (MASKED) x[r][e] = ((t + r) * 32 + 16 * (e >> 3) + 8 * hh + (e & 7)) < lim ? x[r][e] : -INFINITY;
#pragma unroll
        for (int e = e0; e < e0 + 8; e += 2) mx[(e >> 1) & 1] = vmax3(mx[(e >> 1) & 1], x[r][e], x[r][e + 1]);
      } else if constexpr (n == 4) {
        const float m_new = vmax(m_run, xor32_max(vmax(mx[0], mx[1])) * scale_log2e);
        m_use = m_new == -INFINITY ? 0.f : m_new;
        al = __builtin_amdgcn_exp2f(m_run - m_use);       // m_run = -inf -> 0
        m_run = m_new;
      } else {
        constexpr int r = (n - 5) >> 3, e = ((n - 5) & 7) * 2;
#pragma unroll
        for (int k = 0; k < 2; ++k) x[r][e + k] = __builtin_amdgcn_exp2f(fmaf(x[r][e + k], scale_log2e, -m_use));   // masked scores are -inf -> 0
        if constexpr (n > 5) settle(std::integral_constant<int, n - 6>{});
      }
    };
    unrolled<2 * NP>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (i >= 2 * VP && (i - 2 * VP) % KP == 0) clear(t + (i - 2 * VP) / KP + 2, sc[(i - 2 * VP) / KP]);
      const bf16x8 fi = as_bf16x8(f[i % (FRAG_LEAD + 1)]);
      if constexpr (i + FRAG_LEAD < 2 * NP) f[(i + FRAG_LEAD) % (FRAG_LEAD + 1)] = read(i + FRAG_LEAD);
      if constexpr (i < 2 * VP) o[(i % VP) >> 1] = mfma32(fi, p_prev[2 * (i / VP) + (i & 1)], o[(i % VP) >> 1]);
      else sc[(i - 2 * VP) / KP] = mfma32(fi, as_bf16x8(qf[(i - 2 * VP) % KP]), sc[(i - 2 * VP) / KP]);
      constexpr int before = Steps::formed(i - 1), formed = Steps::formed(i);
      if constexpr (i < 5) step(ic);
      unrolled<formed - before>([&](auto k) {
        constexpr int n = before + decltype(k)::value;
        if constexpr (n < 16) step(std::integral_constant<int, 5 + n>{}); else settle(std::integral_constant<int, 15>{});
      });
      unrolled<16>([&](auto kc) {             // rounded, into the registers of the pending P whose last MFMA has been issued
        constexpr int k = decltype(kc)::value, last = ((k >> 3) + 1) * VP - 1;
        if constexpr (k + 1 < formed && (i == last || (i > last && k + 1 >= before))) {
          unsigned v = pack2(x[k >> 3][(k & 7) * 2], x[k >> 3][(k & 7) * 2 + 1]);
          asm volatile("" : "+v"(v));
          w[k >> 2][k & 3] = v;
        }
      });
#pragma unroll
      for (int j = 0; j < PWP; ++j)
        if (i == (2 * j + 1) * NP / PWP) issue(j, t + 4, ps);
      if (LM) __builtin_amdgcn_sched_barrier(0);      // this order is the order of issue (tower: 18 slices of 880 121 us, 123 without; D = 128: 1.5 % slower with it)
    });
    if (!LM) l_run = l_run * al + (psum[0] + psum[1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) p_prev[i] = as_bf16x8(w[i]);
    alpha = al;
  };
  auto rescale = [&] {                                  // alpha is one while a row's maximum stands (x * 1.0f is exact: its bits do not depend on its neighbours)
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f) == 0) return;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
  };

  // K of tiles tb and tb + 1 (the slots of the third pair-stage, free until the loop's first iteration is past its barrier), then two pairs
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int j = 0; j < PK; ++j) {
      const int p = min(j * NWAVE + wave, Im::KPD - 1), row = (p * 64 + lane) / Im::CR, c = (p * 64 + lane) % Im::CR;
      piece(reinterpret_cast<const char*>(kv.k), (unsigned)kv.k_tile, min(tb + r, kv.ntile - 1), kv.k_row,
            (CLAMP ? 0u : (unsigned)row * kv.k_row) + (unsigned)((c ^ Im::kx(row)) * 16), row, lds0 + (unsigned)(4 + r) * Im::SLOT + (unsigned)p * (D == 128 ? 1040 : 1024));
    }
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int j = 0; j < PWP; ++j) issue(j, tb + 2 * k, k);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PWP) : "memory");
  __builtin_amdgcn_s_barrier();
  if (active) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      clear(tb + r, sc[r]);
#pragma unroll
      for (int ks = 0; ks < KP; ++ks) sc[r] = mfma32(as_bf16x8(kfrag(alds + (4 + r) * Im::SLOT, ks)), as_bf16x8(qf[ks]), sc[r]);
    }
  }
  for (int t = tb; t < te; t += 2) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PWP) : "memory");
    __builtin_amdgcn_s_barrier();
    if (active) {
      if (t > tb + 2) rescale();                        // O is zero until then
      if ((t + 2) * 32 > mlim) pair(std::true_type{}, t); else pair(std::false_type{}, t);
    } else {
#pragma unroll
      for (int j = 0; j < PWP; ++j) issue(j, t + 4, st == 0 ? 2 : st - 1);
    }
    st = st == 2 ? 0 : st + 1;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");     // all pieces: no LDS-DMA of this block may land after it has left the CU
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (active) {                // the last pair's P.V: its V^T is in the next pair's slots
    rescale();
#pragma unroll
    for (int i = 0; i < 2 * VP; ++i) o[(i % VP) >> 1] = mfma32(as_bf16x8(vfrag(alds + (2 * st + i / VP) * Im::SLOT, i % VP)), p_prev[2 * (i / VP) + (i & 1)], o[(i % VP) >> 1]);
  }
}

// ------------------------------------------------------------------------------------------------------------------------------
// LLM prefill (causal, GQA): grid = (query tiles, KV heads, key splits); NWAVE waves: wave w < G computes query head hk * G + w, every
// wave feeds the DMA ring.  Tile tables as attn_prefill_kernel: stream slot, first row in q, valid rows (<= 32), cache index of row 0.
// Round 6, two changes of the work mapping (both leave every (row, head)'s arithmetic untouched: bit-identical outputs):
//  * XCD-chunked block order (`xcd_chunks`): the grid is 1-D; work item = (key split, KV head, query tile) with the query tile fastest, and
//    the items are dealt to the 8 XCDs in CONTIGUOUS chunks (block b runs on XCD b % 8 -- observed placement, used for speed only): the
//    query tiles of one stream that read the SAME keys of a (KV head, split) then run on ONE XCD and share its L2.  Before, blockIdx.x
//    = query tile put the 13 tiles of a 386-row chunk on 8 different XCDs, i.e. every K / V byte was pulled into 8 L2s (8 x 386 rows x
//    6.5k keys: 1.4 GB of L2 fills per launch = 3.4 TB/s, all of it LDS-DMA latency in front of the ring's vmcnt waits).
//  * (row, head) pair packing (`pack`): a wave's 32 query columns are 32 consecutive (head, row) PAIRS of the tile's nq x G pairs, head-major
//    (pair p = head_local * nq + row), instead of "wave w = head w, column = row".  With nq = 32 that is the same thing; a ragged tile
//    (386 rows = 12 x 32 + 2) packs its 2 x 7 = 14 pairs into ONE wave instead of running seven waves with two live columns each -- 1/7
//    of the MFMA work for 1/13 of a chunk's blocks.
// __launch_bounds__(.., 2): never the AGPR form of the MFMAs -- the 4-wave instantiation (G <= 4) was built with 512 registers allowed and
// copied O and the scores between AGPRs and VGPRs in every region (144 v_accvgpr_read / write on top of 115 vector instructions; round-6 audit,
// tools/audit_agpr_copies.py); 236 VGPRs now, no copies.
template <int NWAVE>
__global__ __launch_bounds__(NWAVE * 64, 2) void attn_gqa32_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const int32_t* __restrict__ tile_stream,
    const int32_t* __restrict__ tile_q0, const int32_t* __restrict__ tile_nq, const int32_t* __restrict__ tile_pos0,
    bf16_t* const* __restrict__ kv_base, KvLayout lay, int layer, int heads, float scale_log2e, int nsplit,
    float* __restrict__ ws_o, float* __restrict__ ws_ml, int n_tiles, int xcd_chunks, int pack) {
  constexpr int D = 128, KP = 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char alds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hh = lane >> 5;
  const int n_items = n_tiles * lay.n_kv_heads * nsplit;
  int item = blockIdx.x;
  if (xcd_chunks) item = (int)(blockIdx.x & 7) * ((n_items + 7) >> 3) + (int)(blockIdx.x >> 3);
  if (item >= n_items) return;                           // (the grid is rounded up to 8 chunks; the whole block leaves before any barrier)
  const int grp = item % n_tiles, hk = (item / n_tiles) % lay.n_kv_heads, split = item / (n_tiles * lay.n_kv_heads);
  const int G = heads / lay.n_kv_heads;
  const int strm = tile_stream[grp], q0 = tile_q0[grp], nq = tile_nq[grp], pos0 = tile_pos0[grp];
  // this lane's (head, row) pair
  const int pairs = nq * G;
  const int pidx = min(wave * 32 + col, pairs - 1);      // clamped: surplus columns compute a valid pair and are not stored
  const int hl = pack ? pidx / nq : min(wave, G - 1);
  const int qr = pack ? pidx - hl * nq : min(col, nq - 1);
  const int h = hk * G + hl;
  const bool active = pack ? wave * 32 < pairs : wave < G;
  const bool valid = pack ? wave * 32 + col < pairs : (wave < G && col < nq);
  const bf16_t* base = kv_base[strm] + (size_t)layer * lay.layer_stride();
  const bf16_t* kbase = base + (size_t)hk * lay.head_stride();
  const bf16_t* vbase = base + lay.kv_stride() + (size_t)hk * lay.head_stride();
  const int nkeys = pos0 + nq, ntile = (nkeys + 31) / 32;
  const int per = (ntile + nsplit - 1) / nsplit;
  const int tb = nsplit > 1 ? min(ntile, split * per) : 0;
  const int te = nsplit > 1 ? min(ntile, tb + per) : ntile;
  const int ldq = heads * D;
  const int key_limit = pos0 + qr + 1;                   // causal, bottom-right aligned: keys 0 .. pos (inclusive)

  // Q^T fragments (B operand of K . Q^T), resident for the whole key loop: Q[row qr][d = ks * 16 + hh * 8 .. + 8]
  u32x4 qf[KP];
  {
    const bf16_t* qp = q + (size_t)(q0 + qr) * ldq + h * D + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) qf[ks] = ld16(qp + ks * 16);
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) settle_load(qf[ks]);     // before the first LDS-DMA piece (common.h: glds16)
  }

  // The KV cache is allocated in whole 32-key tiles, so the rows of the last (partial) tile exist and are masked.
  Kv32 kv; kv.k = kbase; kv.v = vbase; kv.k_row = D * 2; kv.v_row = 64; kv.k_tile = 32 * D * 2; kv.v_tile = D * 64; kv.ntile = ntile; kv.nkeys = nkeys;

  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  int min_limit = key_limit;                             // wave-wide minimum of the key limits: tiles entirely below it need no mask
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) min_limit = min(min_limit, __shfl_xor(min_limit, off, 64));
  attn32_key_loop<D, D, NWAVE, false>(alds, kv, qf, tb, te, min(min_limit, te * 32), min(key_limit, te * 32), scale_log2e, active, lane, wave, hh, o, m_run, l_run);
  if (!active) return;

  float l = xor32_sum(l_run);
  if (nsplit > 1) {      // partial (o, m, l) of this key split; attn_prefill_combine_kernel merges them
    if (valid) {
      const size_t slot = ((size_t)(q0 + qr) * heads + h) * nsplit + split;
      float* op = ws_o + slot * D;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          *reinterpret_cast<f32x4*>(op + dt * 32 + 8 * r4 + 4 * hh) =
              (f32x4){o[dt][4 * r4], o[dt][4 * r4 + 1], o[dt][4 * r4 + 2], o[dt][4 * r4 + 3]};
      if (hh == 0) { ws_ml[slot * 2] = m_run; ws_ml[slot * 2 + 1] = l; }
    }
    return;
  }
  const float inv = 1.f / l;
  if (valid) {
    bf16_t* op = out + (size_t)(q0 + qr) * ldq + h * D;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        st8(op + dt * 32 + 8 * r4 + 4 * hh, (u32x2){pack2(o[dt][4 * r4] * inv, o[dt][4 * r4 + 1] * inv),
                                                   pack2(o[dt][4 * r4 + 2] * inv, o[dt][4 * r4 + 3] * inv)});
  }
}

// ------------------------------------------------------------------------------------------------------------------------------
// ViT attention (Q2VL:375-417: non-causal inside each temporal slice, d = 80) on the same key loop.  grid = (groups of NWAVE x 32
// query rows of ONE segment, heads): wave w owns the 32 rows q0 + 32 w of the group, all waves share the segment's K / V^T tiles of
// this head through the ring.  d = 80 is 5 k-steps of the 32x32x16 MFMA for K.Q^T (no padding; the 16x16x32 kernel pads 80 -> 96)
// and 3 d-tiles for O^T (the third half empty: ones, see LM).  qkv = [P, 3E] with q, k rotated in place,
// vt = V blocked-transposed [head][32-key block][80][32] (vit_rope_vt_kernel); keys past the segment end are masked, and the K rows of
// the last (partial) tile are clamped into the segment (the next segment's rows are NOT part of this attention).
// NWAVE 4: two blocks share a compute unit (67,584 bytes of LDS each), so one's ends hide behind the other, and 880 rows are 7 groups of 128 instead of 4 of 256:
// 18 slices of 880 132 us against 151, 40 of 400 87 / 93, 8 of 1,456 132 / 128 (one card, in turn).  NWAVE 8 serves calls under a grid cap (one block a unit).
template <int NWAVE>
__global__ __launch_bounds__(NWAVE * 64, 2) void attn_vit32_kernel(
    const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ vt, bf16_t* __restrict__ out, const int32_t* __restrict__ grp_seg,
    const int32_t* __restrict__ grp_q0, const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_len,
    const int32_t* __restrict__ seg_blk_start, int heads, int total_blocks, float scale_log2e, int n_groups, int xcd_chunks) {
  constexpr int D = 80, KP = 5, DT = 3;
  using Im = Attn32Image<D, D>;
  extern __shared__ __attribute__((aligned(16))) unsigned char alds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hh = lane >> 5;
  // V^T rows 80..95 of the third d-tile do not exist: ones in every slot (the DMA copies rows 0..79), so O^T rows 80..95 = sum of P
  for (int i = threadIdx.x; i < 6 * 64; i += NWAVE * 64)
    *reinterpret_cast<u32x4*>(alds + (i >> 6) * Im::SLOT + Im::KB + 80 * 64 + (i & 63) * 16) = (u32x4){0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // before the key loop's first barrier
  // one (group, head) per block, or a persistent walk under the grid cap (gemm.hip: g_grid_cap): virtual block vb = head * n_groups + group.
  // xcd_chunks (round 6): the virtual blocks are dealt to the 8 XCDs in contiguous chunks (block b runs on XCD b % 8: speed only), so the
  // ~6 row groups that read the same segment's K / V of one head share ONE L2 instead of landing on six
  const int nvb = n_groups * heads, c8 = (nvb + 7) >> 3, vlimit = xcd_chunks ? 8 * c8 : nvb;
  for (int vb0 = blockIdx.x; vb0 < vlimit; vb0 += gridDim.x) {
  const int vb = xcd_chunks ? (vb0 & 7) * c8 + (vb0 >> 3) : vb0;
  if (vb >= nvb) break;
  const int h = vb / n_groups, grp = vb - h * n_groups, E = heads * D, ld = 3 * E;
  const int sg = grp_seg[grp], q0 = grp_q0[grp] + wave * 32;
  const int s0 = seg_start[sg], sl = seg_len[sg];
  const bf16_t* kbase = qkv + (size_t)s0 * ld + E + h * D;
  const bf16_t* vbase = vt + ((size_t)h * total_blocks + seg_blk_start[sg]) * (D * 32);
  const int nkeys = sl, ntile = (nkeys + 31) / 32;
  const bool active = q0 < sl;
  const int nq = max(0, min(32, sl - q0));
  const int qrow = min(q0 + min(col, max(nq - 1, 0)), sl - 1);      // clamped: inactive waves / surplus columns read a valid row

  u32x4 qf[KP];
  {
    int hq = hh;          // opaque: formed for every (group, head), not kept in registers through the key loop
    asm volatile("" : "+v"(hq));
    const bf16_t* qp = qkv + (size_t)(s0 + qrow) * ld + h * D + hq * 8;
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) qf[ks] = ld16(qp + ks * 16);
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) settle_load(qf[ks]);     // before the first LDS-DMA piece (common.h: glds16)
  }
  Kv32 kv; kv.k = kbase; kv.v = vbase; kv.k_row = (unsigned)ld * 2; kv.v_row = 64; kv.k_tile = (size_t)64 * ld; kv.v_tile = D * 64; kv.ntile = ntile; kv.nkeys = nkeys;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  attn32_key_loop<D, D, NWAVE, true, false, true>(alds, kv, qf, 0, ntile, sl, sl, scale_log2e, active, lane, wave, hh, o, m_run, l_run);
  const float l = o[2][8];                               // row 80 + 4 hh of O^T, every one of rows 80..95 holds the sum over ALL keys
  if (active && col < nq) {
    const float inv = 1.f / l;
    bf16_t* op = out + (size_t)(s0 + q0 + col) * E + h * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int d = dt * 32 + 8 * r4 + 4 * hh;
        if (d < D)
          st8(op + d, (u32x2){pack2(o[dt][4 * r4] * inv, o[dt][4 * r4 + 1] * inv), pack2(o[dt][4 * r4 + 2] * inv, o[dt][4 * r4 + 3] * inv)});
      }
  }
  if (vb0 + (int)gridDim.x < vlimit) __syncthreads();     // the next (group, head)'s DMA ring reuses the stages
  }
}

template <int NWAVE>
static void vit32_launch_t(const bf16_t* qkv, const bf16_t* vt, bf16_t* out, const int32_t* grp_seg, const int32_t* grp_q0, const int32_t* seg_start,
                           const int32_t* seg_len, const int32_t* seg_blk_start, int n_groups, int heads, int total_blocks, float scale_log2e, hipStream_t st) {
  constexpr size_t lds = Attn32Image<80, 80>::BYTES;
  static DeviceOnce once;   // per instantiation
  if (once.first()) (void)hipFuncSetAttribute((const void*)attn_vit32_kernel<NWAVE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  const long nvb = (long)n_groups * heads;
  const int cap = get_grid_cap();
  static const int xcd = [] { const char* v = getenv("LCC_ATTN32_XCD"); return v ? atoi(v) : 1; }();      // A/B: 0 = virtual block = physical block
  const long nb = (cap > 0 && nvb > cap) ? cap : (xcd ? (nvb + 7) / 8 * 8 : nvb);      // (the cap is a multiple of 8: gemm.hip set_grid_cap)
  attn_vit32_kernel<NWAVE><<<dim3((unsigned)nb), dim3(NWAVE * 64), lds, st>>>(
      qkv, vt, out, grp_seg, grp_q0, seg_start, seg_len, seg_blk_start, heads, total_blocks, scale_log2e, n_groups, xcd);
}
int attn_vit32_launch(const bf16_t* qkv, const bf16_t* vt, bf16_t* out, const int32_t* grp_seg, const int32_t* grp_q0,
                      const int32_t* seg_start, const int32_t* seg_len, const int32_t* seg_blk_start, int n_groups, int heads,
                      int total_blocks, float scale_log2e, hipStream_t st, int group_rows) {
  if (n_groups <= 0) return 0;
  if (group_rows != 256 && group_rows != 128) return LCC_ERR_ARG;
  // group_rows 256: 8 waves x 32 rows per block; 128: 4 waves, two blocks a compute unit
  auto go = [&](auto nw) { vit32_launch_t<decltype(nw)::value>(qkv, vt, out, grp_seg, grp_q0, seg_start, seg_len, seg_blk_start, n_groups, heads, total_blocks, scale_log2e, st); };
  if (group_rows == 256) go(std::integral_constant<int, 8>{}); else go(std::integral_constant<int, 4>{});
  g_launch_counts[LC_ATTN_VIT32] += 1;
  return 0;
}

// Query rows per tile.  With the (row, head) pair packing a block serves nq x G pairs in NWAVE x 32 columns, so a tile may hold up to
// NWAVE * 32 / G rows: 36 at G = 7 (252 of the 256 columns busy -- with 32-row tiles the eighth wave of every block idles, and a block's time
// is that of its busiest SIMD either way), 42 at G = 6, 32 at G = 8 or 4.  LCC_ATTN32_TILE_ROWS (A/B, read once): 32 = the round-3..6 tiles.
static int attn32_pack_on() {
  static const int pack = [] { const char* v = getenv("LCC_ATTN32_PACK"); return v ? atoi(v) : 1; }();
  return pack;
}
int attn32_max_tile_rows(int G) {
  if (G < 1 || G > 8 || !attn32_pack_on()) return 32;
  return std::min(64, ((G <= 4 ? 4 : 8) * 32) / G);
}
int attn32_tile_rows(int G) {
  static const int forced = [] { const char* v = getenv("LCC_ATTN32_TILE_ROWS"); return v ? atoi(v) : 0; }();
  const int mx = attn32_max_tile_rows(G);
  return forced >= 16 ? std::min(forced, mx) : mx;
}

// Tile height and key-split count of one prefill launch, planned TOGETHER (host logic only: lcc_debug_attn_plan pins it on the CPU).
// One 8-wave block per CU and (tile, KV head, split); a block's time is proportional to its keys and does not depend on how many of its
// waves work.  Cost of a candidate (tile rows, k splits) in units of one unsplit block's time:
//     ceil(tiles x kv_heads x k / cus) / k          rounds of blocks on the chip x keys per block
//   + k x (0.01 + 200 / max_kv)                     what a split costs: its fp32 partials written and merged (~4 us per split against ~0.02 us
//                                                   per key of a block), and a small preference for fewer splits between near-ties
// k <= 8 with >= 8 key tiles per split, and only for S <= 1024 rows (the partial buffers of carve_llm).  The model ranks every measured
// configuration of profiles/r06/attn_tall_tiles_ab.jsonl / attn_tall_tiles_splits_probe.jsonl in the measured order:
//   1 chunk  (386 rows, 6.2k keys): (36, 5) 65.4 us < (36, 4) 72.2 ~ (32, 4) 73.4 << (32, 1) 181
//   2 chunks: (32, 2) 113.7 < (36, 2) 116 < (36, 8) 125.8 ~ (36, 4) 127.4 < (32, 7) 129 < (36, 3) 152.7 < (32, 1) 176
//             (rounds 3-6 maximised "filled fraction of the last round" instead and ran 2-chunk batches at (32, 7): +13 %)
//   3 chunks: (36, 3) 163 < (32, 1) 179 < (36, 4) 190 < (32, 2) 206 < (36, 2) 214  (the engine runs (32, 1) there: 1,158 rows > 1,024)
//   4 / 8 chunks (no split above 1,024 rows): (32, 1) = (36, 1) within 1 %: ties keep 32 rows; 8 first turns: (36, 1) 132 < (32, 1) 140 (4 vs 5 rounds)
void attn32_plan(const int* n_new, int n_streams, int max_kv, int G, int n_kv_heads, int cus, int* tile_rows, int* splits) {
  long S = 0;
  for (int b = 0; b < n_streams; ++b) S += n_new[b];
  const int ks_cap = S <= 1024 ? std::max(1, std::min(8, (max_kv / 32) / 8)) : 1;
  const float per_split = 0.01f + 200.f / (float)std::max(max_kv, 32);
  const int tall = attn32_tile_rows(G);
  float best = 1e30f;
  *tile_rows = 32; *splits = 1;
  for (int pass = 0; pass < (tall > 32 ? 2 : 1); ++pass) {           // 32-row tiles first: they win ties
    const int rows = pass == 0 ? 32 : tall;
    long tiles = 0;
    for (int b = 0; b < n_streams; ++b) tiles += (n_new[b] + rows - 1) / rows;
    const long base = tiles * n_kv_heads;
    for (int k = 1; k <= ks_cap; ++k) {
      const float cost = (float)((base * k + cus - 1) / cus) / (float)k + per_split * (float)k;
      if (cost < best - 1e-6f) { best = cost; *tile_rows = rows; *splits = k; }
    }
  }
}

// launcher: tiles of <= attn32_max_tile_rows(G) rows; the caller (attention.hip: attn_prefill_bf16) runs the split merge
int attn_prefill32_launch(const bf16_t* q, bf16_t* out, const int32_t* tile_stream, const int32_t* tile_q0, const int32_t* tile_nq,
                          const int32_t* tile_pos0, bf16_t* const* kv_base, KvLayout lay, int layer, int n_tiles, int n_q_heads,
                          int nsplit, float* ws_o, float* ws_ml, float scale_log2e, hipStream_t st) {
  const int G = n_q_heads / lay.n_kv_heads;
  if (G < 1 || G > 8 || lay.head_dim != 128) return LCC_ERR_SHAPE;
  constexpr size_t lds = Attn32Image<128, 128>::BYTES;
  static DeviceOnce once;
  if (once.first()) {
    (void)hipFuncSetAttribute((const void*)attn_gqa32_kernel<8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)hipFuncSetAttribute((const void*)attn_gqa32_kernel<4>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  }
  const int S = nsplit > 1 ? nsplit : 1;
  // LCC_ATTN32_XCD / LCC_ATTN32_PACK (A/B, read once): 0 = the round-3..5 work mapping (blockIdx = tile / KV head / split; wave = head)
  static const int xcd = [] { const char* v = getenv("LCC_ATTN32_XCD"); return v ? atoi(v) : 1; }();
  const int pack = attn32_pack_on();
  const long n_items = (long)n_tiles * lay.n_kv_heads * S;
  const dim3 grid((unsigned)(xcd ? ((n_items + 7) / 8) * 8 : n_items));
  if (G <= 4)
    attn_gqa32_kernel<4><<<grid, dim3(256), lds, st>>>(q, out, tile_stream, tile_q0, tile_nq, tile_pos0, kv_base, lay, layer, n_q_heads,
                                                       scale_log2e, S, ws_o, ws_ml, n_tiles, xcd, pack);
  else
    attn_gqa32_kernel<8><<<grid, dim3(512), lds, st>>>(q, out, tile_stream, tile_q0, tile_nq, tile_pos0, kv_base, lay, layer, n_q_heads,
                                                       scale_log2e, S, ws_o, ws_ml, n_tiles, xcd, pack);
  return 0;
}

// ------------------------------------------------------------------------------------------------------------------------------
// Causal multi-head attention (one KV head per query head) over freshly formed keys and transposed values -- the prefill form of latent
// attention (latent.hip).  Work item = (head, group of up to 256 rows of one stream), wave w owns rows 32 w ..; the eight waves share the
// head's K / V^T tiles through the ring.  A wave whose rows end before the group's last key tile runs that tile fully masked.  Items are
// dealt to the XCDs in contiguous chunks, groups fastest (and from the back: the long ones first), so the groups that read the same keys share
// an L2.  The per-head output factor `gate` is applied before the one rounding to bf16.
// ------------------------------------------------------------------------------------------------------------------------------
// SLOTS: keys and values out of the slots' arenas, shared by the query heads of a KV head, and a distance bias per head (kernels.h: MhaArgs).
template <int DK, int DV, bool SLOTS>
__global__ __launch_bounds__(512, 2) void attn_mha32_kernel(MhaArgs a) {
  constexpr int NWAVE = 8, KP = DK / 16, DT = DV / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char alds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hh = lane >> 5;
  const int n_items = a.n_groups * a.heads;
  const int item = (int)(blockIdx.x & 7) * ((n_items + 7) >> 3) + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= ((n_items + 7) >> 3) || item >= n_items) return;      // the whole block leaves before any barrier
  const int h = item / a.n_groups, grp = a.n_groups - 1 - (item - h * a.n_groups);
  const int q0 = a.grp_q0[grp], nq = a.grp_nq[grp], pos0 = a.grp_pos0[grp], key0 = SLOTS ? 0 : a.grp_key0[grp];
  const int ldq = a.heads * DK;
  const bool active = wave * 32 < nq;
  const int qr = min(wave * 32 + col, nq - 1);           // clamped: surplus columns compute a valid row and are not stored
  const bool valid = wave * 32 + col < nq;
  const int ntile = (pos0 + nq + 31) / 32;               // the keys are stored in whole 32-key tiles (zero-filled)
  const int ldk = SLOTS ? DK : ldq, ldv = SLOTS ? 32 : a.ldv;
  const bf16_t *kbase, *vbase;
  if (SLOTS) {
    const bf16_t* arena = a.kv_base[a.grp_slot[grp]];
    const int kvh = h / (a.heads / a.kv_heads);
    kbase = arena + a.k_off + (size_t)kvh * a.lmax * DK;
    vbase = arena + a.v_off + (size_t)kvh * a.lmax * DV;
  } else {
    kbase = a.k + (size_t)key0 * ldq + h * DK;
    vbase = a.vt + (size_t)h * DV * a.ldv + key0;
  }

  u32x4 qf[KP];
  {
    const bf16_t* qp = a.q + (size_t)(q0 + qr) * ldq + h * DK + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) qf[ks] = ld16(qp + ks * 16);
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) settle_load(qf[ks]);     // before the first LDS-DMA piece (common.h: glds16)
  }
  // the key loop takes a positive scale: a negative one turns the sign of q, none at all leaves the bias alone
  float scale = a.scale_log2e;
  if (scale <= 0.f) {
#pragma unroll
    for (int ks = 0; ks < KP; ++ks)
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[ks][e] = scale < 0.f ? qf[ks][e] ^ 0x80008000u : 0u;
    scale = scale < 0.f ? -scale : 1.f;
  }
  Kv32 kv; kv.k = kbase; kv.v = vbase; kv.k_row = (unsigned)ldk * 2; kv.v_row = (unsigned)ldv * 2; kv.k_tile = (size_t)64 * ldk; kv.v_tile = SLOTS ? (size_t)DV * 64 : 64;
  kv.ntile = ntile; kv.nkeys = pos0 + nq;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const int key_limit = pos0 + qr + 1;
  int min_limit = pos0 + min(wave * 32, nq - 1) + 1;            // of the wave's first row
  asm volatile("" : "+v"(min_limit));
  const float slope = SLOTS && a.slope ? a.slope[h] : 0.f;
  attn32_key_loop<DK, DV, NWAVE, false, SLOTS>(alds, kv, qf, 0, ntile, min_limit, key_limit, scale, active, lane, wave, hh, o, m_run, l_run, slope, pos0 + qr);
  if (!active) return;
  const float l = xor32_sum(l_run);
  if (valid) {
    const float f = (a.gate ? a.gate[(size_t)(q0 + qr) * a.heads + h] : 1.f) / l;
    bf16_t* op = a.out + (size_t)(q0 + qr) * a.ldo + h * DV;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        st8(op + dt * 32 + 8 * r4 + 4 * hh, (u32x2){pack2(o[dt][4 * r4] * f, o[dt][4 * r4 + 1] * f), pack2(o[dt][4 * r4 + 2] * f, o[dt][4 * r4 + 3] * f)});
  }
}
template <int DK, int DV, bool SLOTS>
static void mha32_go(const MhaArgs& a, hipStream_t st) {
  constexpr size_t lds = Attn32Image<DK, DV>::BYTES;
  static DeviceOnce once;   // per instantiation
  if (once.first()) (void)hipFuncSetAttribute((const void*)attn_mha32_kernel<DK, DV, SLOTS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  const long n_items = (long)a.n_groups * a.heads;
  attn_mha32_kernel<DK, DV, SLOTS><<<dim3((unsigned)((n_items + 7) / 8 * 8)), dim3(512), lds, st>>>(a);
}
template <bool SLOTS>
static int mha32_pick(const MhaArgs& a, hipStream_t st) {
  if (a.dim == 128 && a.vdim == 128) mha32_go<128, 128, SLOTS>(a, st);
  else if (a.dim == 64 && a.vdim == 64) mha32_go<64, 64, SLOTS>(a, st);
  else if (a.dim == 64 && a.vdim == 128) mha32_go<64, 128, SLOTS>(a, st);
  else if (a.dim == 128 && a.vdim == 64) mha32_go<128, 64, SLOTS>(a, st);
  else return LCC_ERR_SHAPE;
  return 0;
}
int attn_mha32_launch(const MhaArgs& a, hipStream_t st) { return a.grp_slot ? mha32_pick<true>(a, st) : mha32_pick<false>(a, st); }

}  // namespace lcc
