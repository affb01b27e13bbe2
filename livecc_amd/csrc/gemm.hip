// bf16 GEMMs of the LiveCC hot path on gfx950 (MI355X):  C[M,N] = A[M,K] * W[N,K]^T  (+bias, +epilogue)
//
// W keeps the nn.Linear layout [N,K] (K contiguous) so that both MFMA operands are read as 8 contiguous
// bf16 (16 bytes) per lane.  fp32 accumulation, one rounding to bf16 at the points where HF rounds.
//
//  * gemm_walk_kernel    : M >= 17, packed W, K % 64 == 0 (LLM prefill, ViT).  MFMA-bound.  8 waves, BM x 256 x 64 tile
//                          (BM 256 / 192 / 160 / 128), LDS-DMA for both operands; one block a compute unit, the DMA ring runs on from tile to tile.
//  * gemm_vit_kernel     : the same pipeline, a tile a block, with the vision q|k|v epilogues (few patches: gemm_strip_kernel, gemm_mid_kernel).
//  * gemm_big_kernel     : the same tiles one a block, both waves of a SIMD in step: 128-row tiles of one round.
//  * gemm_walk_vh_kernel : the walk over row tiles of 256 / 272 / 288 rows (no ragged last row tile).
//  * gemm_vh_kernel      : row tiles of 128 / 144 rows, split-K slabs of one streaming chunk.
//  * gemm_tall_kernel    : one block row covers all of M (up to 448 rows: gate/up of one streaming chunk or of a few short ones; wide products of 257 rows and more).
//  * gemm_strip_kernel   : shapes with few 256-column tiles.  64x128x64 tile, 4 waves, weights straight into registers, idle compute units fetch them ahead.
//  * gemm_mid_kernel     : the same shapes with more rows.  128x128x64 tile, 8 waves, 4-stage LDS-DMA ring.
//  * gemm_glds_kernel /   : row-major W, K % 64 != 0.  64x128x64 (128x128x64) tile, 4 waves,
//    gemm_tiled_kernel     LDS-DMA 3-stage ring / register-staged double buffer with an XOR swizzle, XCD-aware block remap.
//  * gemv_skinny_kernel  : M <= 64 (decode, lm_head; MG = ceil(M / 16) activation fragments per weight fragment).  HBM-bound weight streaming.  4 waves per block share 16 (32, 64) W rows,
//                          each wave a slice of K; W fragments go straight from HBM into the MFMA operand registers (no LDS
//                          round trip - the operand is used once), split-K partial sums as fp32 slabs that the consumer reduces.
//  * gemv_w8_kernel      : the same for fp8-e4m3 weights + fp32 row scales (PACKED8 order), e4m3 -> bf16 exactly in registers.
//
// Replaces: every nn.Linear / Conv3d of HF modeling_qwen2_vl.py on the path
//   (PatchEmbed 251-274, VisionAttention.qkv/proj 349-350, VisionMlp 293-301, PatchMerger 277-290,
//    Qwen2VLAttention q/k/v/o_proj 501-504, Qwen2MLP 453-466, lm_head 1218/1323).
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"
#include "tail_ops.h"

namespace lcc {

constexpr int STRIP_STAGES = 6;      // k-tiles a block of gemm_strip_kernel holds
__device__ unsigned int lcc_zero_page[256];  // 1 KB of zeros: operand source of absent K chunks (address select, no branch)

// Grid cap (round 5): while it is set (engine_vit.hip sets it around a vision-tower call that runs on the side stream UNDER another turn's
// decode steps), the MFMA-bound tile kernels launch at most `cap` workgroups and walk their tiles persistently (tile = block, block +
// grid, ...), so that they occupy `cap` of the 256 CUs instead of all of them.  Why: a resident 8-wave GEMM block (2 x 208-216 VGPRs per
// SIMD, 128-140 KB of LDS) leaves room for ONE weight-streaming decode wave per SIMD where five fit on a free CU -- with the tower spread
// over every CU the HBM-bound decode kernels lose their memory-level parallelism and the "overlapped" tower simply adds its own duration
// to the decode steps (8 streams: 4.88 vs 3.68 ms per step while a 20-ms tower runs; 1 stream: 3.23 vs 2.95 ms).  Half the CUs stream the
// weights at the full HBM rate.  A multiple of 8 (virtual block id and physical block id then agree on the XCD).
// thread_local: the cap belongs to the host thread that is inside lcc_vit_encode -- a second thread launching prefill GEMMs
// meanwhile is not capped, and two engines with different caps do not race.
static thread_local int g_grid_cap = 0;
void set_grid_cap(int cap) { g_grid_cap = cap <= 0 ? 0 : std::max(8, cap & ~7); }
int get_grid_cap() { return g_grid_cap; }
static inline unsigned capped_grid(long nblk) { return (unsigned)((g_grid_cap > 0 && nblk > g_grid_cap) ? g_grid_cap : nblk); }

// epilogue shared by the tiled kernels.  acc[i][j][r] = C[mbase + i*16 + li][nbase + j*16 + g*4 + r] (swapped operands).
template <int EPI, int MT, int NT, int AM = MT, int AN = NT>   // the first MT x NT tiles of an AM x AN accumulator array
LCC_DEVICE void tile_epilogue(const f32x4 (&acc)[AM][AN], int mbase, int nbase, int ocbase, int li, int g,
                              const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
                              bf16_t* __restrict__ C, int ldc, int M, int N, float* __restrict__ partial,
                              const float* __restrict__ wscale) {
  // per-output-row dequantisation scale of fp8 weights (1.0 for bf16 weights: x * 1.0 is exact)
  f32x4 sc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) sc[j] = (f32x4){1.f, 1.f, 1.f, 1.f};
  if (wscale != nullptr) {
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = *reinterpret_cast<const f32x4*>(wscale + min(nbase + j * 16 + g * 4, N - 4));
  }
  // Loads (bias: once per column group; residual: NT per row tile) are issued unconditionally from clamped addresses and
  // back to back, so that they overlap instead of one L2 round trip per (row tile, column group); only the stores are
  // predicated on the M / N edges.
  u32x2 bv[NT];
  if (EPI != EPI_PARTIAL && EPI != EPI_SWIGLU) {
#pragma unroll
    for (int j = 0; j < NT; ++j) bv[j] = (u32x2){0u, 0u};
    if (bias != nullptr) {
#pragma unroll
      for (int j = 0; j < NT; ++j) bv[j] = ld8(bias + min(nbase + j * 16 + g * 4, N - 4));
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = mbase + i * 16 + li;
    const bool mok = m < M;
    const int mc = min(m, M - 1);
    if (EPI == EPI_PARTIAL) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n = nbase + j * 16 + g * 4;
        if (mok && n < N) *reinterpret_cast<f32x4*>(partial + ((size_t)blockIdx.y * M + m) * N + n) = acc[i][j] * sc[j];
      }
    } else if (EPI == EPI_SWIGLU) {
#pragma unroll
      for (int j = 0; j < NT; j += 2) {
        const int n = nbase + j * 16 + g * 4;  // column in the interleaved [gate16|up16] space
        const int oc = ocbase + (j / 2) * 16 + g * 4;
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float gate = rbf(acc[i][j][r] * sc[j][r]), up = rbf(acc[i][j + 1][r] * sc[j + 1][r]);
          o[r] = silu_bf16(gate) * up;
        }
        if (mok && n < N) st8(C + (size_t)m * ldc + oc, (u32x2){pack2(o[0], o[1]), pack2(o[2], o[3])});
      }
    } else {
      u32x2 rv[NT];
      if (EPI == EPI_RESIDUAL) {
#pragma unroll
        for (int j = 0; j < NT; ++j) rv[j] = ld8(residual + (size_t)mc * ldr + min(nbase + j * 16 + g * 4, N - 4));
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n = nbase + j * 16 + g * 4;
        float v[4] = {acc[i][j][0] * sc[j][0] + lo2f(bv[j].x), acc[i][j][1] * sc[j][1] + hi2f(bv[j].x), acc[i][j][2] * sc[j][2] + lo2f(bv[j].y),
                      acc[i][j][3] * sc[j][3] + hi2f(bv[j].y)};
        rbf2(v[0], v[1]); rbf2(v[2], v[3]);
        if (EPI == EPI_QUICK_GELU) {
          quick_gelu2(v[0], v[1]); quick_gelu2(v[2], v[3]);
        } else if (EPI == EPI_GELU_ERF) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = gelu_erf_bf16(v[r]);
        } else if (EPI == EPI_RESIDUAL) {
          v[0] += lo2f(rv[j].x); v[1] += hi2f(rv[j].x); v[2] += lo2f(rv[j].y); v[3] += hi2f(rv[j].y);
        }
        if (mok && n < N) st8(C + (size_t)m * ldc + n, (u32x2){pack2(v[0], v[1]), pack2(v[2], v[3])});
      }
    }
  }
}

// The bias / GELU / residual epilogues with 16-byte accesses of whole rows: 64 rows of a wave's columns at a time go through LDS of its own
// (`lds`, 64 x NT x 32 bytes, wave-private: no barrier; the caller has made sure that nobody reads or DMAs into it any more), so that a store
// covers 128 (NT = 2: 64) consecutive bytes of a row instead of 32, and a residual arrives in the same pieces, the next 64 rows' under the
// stores of these -- the plain form waits for its residual row tile by row tile.  Same values, same roundings.  16-byte chunk c of row r sits
// at c ^ (r >> 1 & 7) (NT = 2: c ^ (r >> 2 & 3)): writes and reads spread over the banks.
// The epilogue is a large part of a short product.  15840 x 5120 with K = 64, plain -> here: bias 55 -> 38 us, quick GELU 71 -> 57 (with the
// shorter activation), residual 130 -> 77; 15840 x 1280 with residual 29 -> 20.  SwiGLU (half the bytes, bound by its arithmetic) measured
// 44.4 / 44.8 and keeps the plain form.
// Needs C and the residual in rows of 16-byte pieces, and a bias that scalar loads can read (wide_rows).
template <int EPI>
LCC_DEVICE bool wide_rows(const bf16_t* C, int ldc, const bf16_t* bias, const bf16_t* residual, int ldr) {
  if (EPI == EPI_PARTIAL || EPI == EPI_SWIGLU) return false;
  return (ldc & 7) == 0 && ((uintptr_t)bias & 3) == 0 && ((uintptr_t)C & 15) == 0 && (EPI != EPI_RESIDUAL || ((ldr & 7) == 0 && ((uintptr_t)residual & 15) == 0));
}
// Four bf16 bias values of columns n .. n + 15 a lane group g owns (n uniform in the wave): through the scalar unit, which has a counter of its own --
// a vector load here would also wait for the LDS-DMA pieces of a walking kernel's next tile.
LCC_DEVICE u32x2 bias_of_group(const bf16_t* bias, int n, int g) {
  typedef const __attribute__((address_space(4))) unsigned* sptr;
  const sptr p = (sptr)(uintptr_t)(bias + __builtin_amdgcn_readfirstlane(n));
  const unsigned x0 = p[0], y0 = p[1], x1 = p[2], y1 = p[3], x2 = p[4], y2 = p[5], x3 = p[6], y3 = p[7];
  const bool odd = (g & 1) != 0, high = (g & 2) != 0;
  return (u32x2){high ? (odd ? x3 : x2) : (odd ? x1 : x0), high ? (odd ? y3 : y2) : (odd ? y1 : y0)};
}
template <int EPI, int MT, int NT, int GRT = 4>                    // GRT: row tiles of a group (lds: GRT x 16 x NT x 32 bytes)
LCC_DEVICE void tile_epilogue_wide(const f32x4 (&acc)[MT][NT], int mbase, int nbase, int lane, const bf16_t* __restrict__ bias,
                                   const bf16_t* __restrict__ residual, int ldr, bf16_t* __restrict__ C, int ldc, int M, int N,
                                   const float* __restrict__ wscale, unsigned char* lds) {
  constexpr int RC = NT * 2, RPS = 64 / RC, RB = RC * 16;          // 16-byte chunks of a row; rows of a store; row bytes
  constexpr int GR = MT < GRT ? MT : GRT;                          // row tiles of a group
  const int li = lane & 15, g = lane >> 4;
  auto swz = [](int r) { return NT == 4 ? (r >> 1) & 7 : (r >> 2) & 3; };
  f32x4 sc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) sc[j] = (f32x4){1.f, 1.f, 1.f, 1.f};
  if (wscale != nullptr) {
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = *reinterpret_cast<const f32x4*>(wscale + min(nbase + j * 16 + g * 4, N - 4));
  }
  u32x2 bv[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) bv[j] = (u32x2){0u, 0u};
  if (bias != nullptr) {
#pragma unroll
    for (int j = 0; j < NT; ++j) bv[j] = bias_of_group(bias, min(nbase + j * 16, N - 16), g);
  }
  constexpr int NS = GR * 16 / RPS;                                // stores of a group
  const int sr = lane / RC, schk = lane & (RC - 1), scol = nbase + schk * 8;          // this lane's row and chunk of a store
  const bool cok = scol < N;
  u32x4 rv[NS];                                                    // residual: a piece of the next group is fetched as this group's is used
  auto load_res = [&](int i0, int q) { return ld16(residual + (size_t)min(mbase + i0 * 16 + q * RPS + sr, M - 1) * ldr + min(scol, N - 8)); };
  if (EPI == EPI_RESIDUAL) {
#pragma unroll
    for (int q = 0; q < NS; ++q) rv[q] = load_res(0, q);
  }
#pragma unroll
  for (int i0 = 0; i0 < MT; i0 += GR) {
    // no row of this group exists (wave-uniform).  Not with a residual: pieces requested and never used would make hipcc wait for all memory in
    // every k-step of the next tile (1200 x 3584, K 18944: 220 -> 240 us)
    if (EPI != EPI_RESIDUAL && mbase + i0 * 16 >= M) break;
    wave_lds_order();          // the last group's rows have been read
#pragma unroll
    for (int ii = 0; ii < GR; ++ii) {
      const int i = i0 + ii, r = ii * 16 + li;
      if (i >= MT) continue;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        float v[4] = {acc[i][j][0] * sc[j][0] + lo2f(bv[j].x), acc[i][j][1] * sc[j][1] + hi2f(bv[j].x),
                      acc[i][j][2] * sc[j][2] + lo2f(bv[j].y), acc[i][j][3] * sc[j][3] + hi2f(bv[j].y)};
        if (EPI == EPI_QUICK_GELU || EPI == EPI_GELU_ERF) { rbf2(v[0], v[1]); rbf2(v[2], v[3]); }      // else: the packing rounds
        if (EPI == EPI_QUICK_GELU) {
          quick_gelu2(v[0], v[1]); quick_gelu2(v[2], v[3]);
        } else if (EPI == EPI_GELU_ERF) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_erf_bf16(v[e]);
        }
        st8(lds + r * RB + (((j * 2 + (g >> 1)) ^ swz(r)) * 16) + (g & 1) * 8, (u32x2){pack2(v[0], v[1]), pack2(v[2], v[3])});
      }
    }
    wave_lds_order();          // rows are read by other lanes than wrote them
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      if (i0 * 16 + q * RPS >= MT * 16) continue;                    // the last group may be shorter
      const int r = q * RPS + sr, m = mbase + i0 * 16 + r;
      u32x4 v = ld16(lds + r * RB + ((schk ^ swz(r)) * 16));
      if (EPI == EPI_RESIDUAL) {
        const u32x4 w = rv[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = pack2(lo2f(v[e]) + lo2f(w[e]), hi2f(v[e]) + hi2f(w[e]));
        if (i0 + GR < MT) rv[q] = load_res(i0 + GR, q);
      }
      if (m < M && cok) st16(C + (size_t)m * ldc + scol, v);
    }
  }
}

// fp32 slabs the same way: GRT x 16 rows of NTG x 64 bytes at a time (lds: GRT x NTG KB, wave-private)
template <int MT, int NT, int GRT = 2, int NTG = NT>
LCC_DEVICE void tile_slab_wide(const f32x4 (&acc)[MT][NT], int mbase, int nbase, int lane, int M, int N, float* __restrict__ partial,
                               const float* __restrict__ wscale, unsigned char* lds) {
  static_assert(NT == 4 && (NTG == 4 || NTG == 2), "64 columns a wave");
  constexpr int RC = NTG * 4, RPS = 64 / RC, RB = RC * 16;         // 16-byte chunks of a row; rows of a store; row bytes
  const int li = lane & 15, g = lane >> 4;
  f32x4 sc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) sc[j] = (f32x4){1.f, 1.f, 1.f, 1.f};
  if (wscale != nullptr) {
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = *reinterpret_cast<const f32x4*>(wscale + min(nbase + j * 16 + g * 4, N - 4));
  }
  auto swz = [](int r) { return NTG == 4 ? r & 15 : (r >> 1) & 7; };
  const int sr = lane / RC, schk = lane & (RC - 1);
#pragma unroll
  for (int i0 = 0; i0 < MT; i0 += GRT) {
    if (mbase + i0 * 16 >= M) break;          // 17 rows of a 128-row tile: one group in four (fp8 steps of 17 to 64 streams)
#pragma unroll
    for (int j0 = 0; j0 < NT; j0 += NTG) {
      const int scol = nbase + j0 * 16 + schk * 4;
      float* out = partial + (size_t)blockIdx.y * M * N + scol;
      wave_lds_order();
#pragma unroll
      for (int ii = 0; ii < GRT; ++ii) {
        if (i0 + ii >= MT) continue;
        const int r = ii * 16 + li;
#pragma unroll
        for (int j = 0; j < NTG; ++j) *reinterpret_cast<f32x4*>(lds + r * RB + (((j * 4 + g) ^ swz(r)) * 16)) = acc[i0 + ii][j0 + j] * sc[j0 + j];
      }
      wave_lds_order();
#pragma unroll
      for (int q = 0; q < GRT * 16 / RPS; ++q) {
        if (i0 * 16 + q * RPS >= MT * 16) continue;
        const int r = q * RPS + sr, m = mbase + i0 * 16 + r;
        const f32x4 v = *reinterpret_cast<const f32x4*>(lds + r * RB + ((schk ^ swz(r)) * 16));
        if (m < M && scol < N) *reinterpret_cast<f32x4*>(out + (size_t)m * N) = v;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// EPI_VIT_QK / EPI_VIT_V (round 4): the vision tower's q|k|v projection writes what its attention kernels read -- q and k rotated (2-D
// RoPE, HF modeling_qwen2_vl.py:225-248) at their natural columns of C, V blocked-transposed into vt[head][32-key block][80][32] -- instead
// of a plain [P, 3E] tensor that vit_rope_vt_kernel re-reads and re-writes (52 us per tower block at 8 streams, 179 MB of traffic).
// One launch of gemm_vit_kernel, or of the 128-column kernels (two of the first, q|k and V apart, where a column tile would hold both) over the `qkv_w_rope` copy of the weight (weights.py: vit_qkv_rope_row_permutation):
//
//  * q|k (N = 2E, EPI_VIT_QK): inside q and inside k every 32 stored rows are [16 first-half channels | their 16 rotation partners],
//    first-half channels enumerated head-major (f = head * 40 + c, c < 40), so a lane's accumulators acc[i][j] / acc[i][j + 1] hold
//    (x[c .. c+3], x[c+40 .. c+43]) of one head: the rotation is register-local (40 % 4 == 0: a lane's four channels never straddle a
//    head).  The block's cos / sin rows (BM x 40 fp32 each, one contiguous piece of the tables) are DMA'd into the LDS the k-loop has
//    finished with: the first version loaded them per (row tile, column pair) from global memory and hipcc put an s_waitcnt vmcnt(0)
//    -- which on gfx9 also waits for the previous iteration's STORES -- into each of the 16 iterations (+15 us on a 137-us GEMM).
//  * V (N = E, EPI_VIT_V): the MFMA operands are swapped (activations as the A operand), so a lane holds 4 consecutive PATCHES of one
//    channel -- 8 contiguous bytes of vt, four lanes = 32 contiguous bytes, the store granularity of the plain epilogue -- and no
//    transpose is needed.  Same products, same k order: same bits.  grp_off[p / 4] = element offset of patch p's key slot inside a
//    (head, channel 0) plane of vt; segment lengths are multiples of 4 (H, W multiples of 28), so a 4-patch group never straddles a
//    segment or a 32-key block.
// ------------------------------------------------------------------------------------------------
template <int MT, int NT>
LCC_DEVICE void vit_qk_epilogue(const f32x4 (&acc)[MT][NT], int mbase, int nbase, int mrow0, int li, int g, const bf16_t* __restrict__ bias,
                                bf16_t* __restrict__ C, int ldc, int M, int N, int E, const float* lcs, const float* lsn) {
  u32x2 b1[NT / 2], b2[NT / 2];
#pragma unroll
  for (int jp = 0; jp < NT / 2; ++jp) {
    b1[jp] = (u32x2){0u, 0u}; b2[jp] = (u32x2){0u, 0u};
    const int n = min(nbase + jp * 32, N - 32);
    if (bias != nullptr) { b1[jp] = ld8(bias + n + g * 4); b2[jp] = ld8(bias + n + 16 + g * 4); }
  }
#pragma unroll
  for (int jp = 0; jp < NT / 2; ++jp) {
    const int j = jp * 2;
    const int n = nbase + j * 16;            // first column of a 32-column group (wave-uniform)
    if (n >= N) continue;
    const int which = n >= E ? 1 : 0;
    const int f = ((n - which * E) >> 5) * 16 + g * 4;
    const int h = f / 40, c = f - h * 40;
    bf16_t* out = C + which * E + h * 80 + c;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = mbase + i * 16 + li;
      const f32x4 cv = *reinterpret_cast<const f32x4*>(lcs + (mrow0 + i * 16 + li) * 40 + c);
      const f32x4 sv = *reinterpret_cast<const f32x4*>(lsn + (mrow0 + i * 16 + li) * 40 + c);
      float x1[4], x2[4], o1[4], o2[4];
      x1[0] = rbf(acc[i][j][0] + lo2f(b1[jp].x)); x1[1] = rbf(acc[i][j][1] + hi2f(b1[jp].x));
      x1[2] = rbf(acc[i][j][2] + lo2f(b1[jp].y)); x1[3] = rbf(acc[i][j][3] + hi2f(b1[jp].y));
      x2[0] = rbf(acc[i][j + 1][0] + lo2f(b2[jp].x)); x2[1] = rbf(acc[i][j + 1][1] + hi2f(b2[jp].x));
      x2[2] = rbf(acc[i][j + 1][2] + lo2f(b2[jp].y)); x2[3] = rbf(acc[i][j + 1][3] + hi2f(b2[jp].y));
#pragma unroll
      for (int r = 0; r < 4; ++r) vit_rope_pair(x1[r], x2[r], cv[r], sv[r], o1[r], o2[r]);
      if (m < M) {
        st8(out + (size_t)m * ldc, (u32x2){pack2(o1[0], o1[1]), pack2(o1[2], o1[3])});
        st8(out + (size_t)m * ldc + 40, (u32x2){pack2(o2[0], o2[1]), pack2(o2[2], o2[3])});
      }
    }
  }
}

// swapped operands: acc[i][j][r] = C[mbase + i*16 + g*4 + r][nbase + j*16 + li]
template <int MT, int NT>
LCC_DEVICE void vit_v_epilogue(const f32x4 (&acc)[MT][NT], int mbase, int nbase, int li, int g, const bf16_t* __restrict__ bias, int M, int N,
                               const VitQkvEpi& vq) {
  int off[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) off[i] = vq.grp_off[min(mbase + i * 16 + g * 4, M - 4) >> 2];
  bf16_t braw[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) braw[j] = 0;
  if (bias != nullptr) {      // one branch around the four loads (a select per column made hipcc wait for each load separately)
#pragma unroll
    for (int j = 0; j < NT; ++j) braw[j] = bias[min(nbase + j * 16 + li, N - 1)];
  }
  float bv[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) bv[j] = bf2f(braw[j]);
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = nbase + j * 16 + li;
    const int nc = min(n, N - 1);
    const int h = nc / 80, c = nc - h * 80;
    bf16_t* base = vq.vt + ((size_t)h * vq.total_blocks * 80 + c) * 32;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const u32x2 o = (u32x2){pack2(acc[i][j][0] + bv[j], acc[i][j][1] + bv[j]), pack2(acc[i][j][2] + bv[j], acc[i][j][3] + bv[j])};
      if (n < N && mbase + i * 16 + g * 4 < M) st8(base + off[i], o);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// tiled GEMM
// ------------------------------------------------------------------------------------------------
template <int BM, int EPI>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, int ldw,
    const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
    bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n, int w_packed,
    float* __restrict__ partial, int kt_per_split) {
  constexpr int BN = 128, BK = 64;
  constexpr int WM = BM / 2;       // wave tile rows (of A)
  constexpr int MT = WM / 16;      // 16-row MFMA tiles per wave in M
  constexpr int NT = 4;            // 16-col MFMA tiles per wave in N (wave tile is WM x 64)
  constexpr int AI = BM * 8 / 256; // 16-byte chunks of the A tile per thread
  constexpr int BI = BN * 8 / 256;
  constexpr int STAGE = (BM + BN) * 8;  // 16-byte units per stage
  __shared__ u32x4 smem[2 * STAGE];

  // XCD-aware remap: hardware places block b on XCD b%8; give every XCD a contiguous range of tile ids
  const int nblk = tiles_m * tiles_n;
  int bid = blockIdx.x;
  {
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  const int tn = bid / tiles_m, tm = bid - tn * tiles_m;  // consecutive ids share the W panel
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, g = lane >> 4;

  // global -> register staging addresses
  const bf16_t* aptr[AI];
  const bf16_t* bptr[BI];
  int aoff[AI], boff[BI];  // LDS offsets (16B units) within a stage
  const int chunk = tid & 7;
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    int row = (tid >> 3) + i * 32;
    int gr = min(m0 + row, M - 1);
    aptr[i] = A + (size_t)gr * lda + chunk * 8;
    aoff[i] = row * 8 + (chunk ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    int row = (tid >> 3) + i * 32;
    int gr = min(n0 + row, N - 1);
    // row-major [N,K]: row*ldw + chunk*8, k-tile stride 64.  packed [N/16][Kp/32][4 g][16 rows][8]: the 1-KB fragment
    // sub-tile of (row tile, 32-k block), k-tile (= two 32-k blocks) stride 1024.
    bptr[i] = w_packed ? W + ((size_t)(gr >> 4) * ((K + 31) >> 5) + (chunk >> 2)) * 512 + (chunk & 3) * 128 + (gr & 15) * 8
                       : W + (size_t)gr * ldw + chunk * 8;
    boff[i] = BM * 8 + row * 8 + (chunk ^ ((row >> 1) & 7));
  }
  const int wstride = w_packed ? 1024 : BK;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  u32x4 ra[AI], rb[BI];
  const bf16_t* zp = reinterpret_cast<const bf16_t*>(lcc_zero_page);
  auto gload = [&](int kt) {
    const int k = kt * BK + chunk * 8;
    const bool ok = k < K;  // K % 8 == 0: a chunk is entirely inside or outside (K tail: load zeros, by address select)
#pragma unroll
    for (int i = 0; i < AI; ++i) ra[i] = ld16(ok ? aptr[i] + kt * BK : zp);
#pragma unroll
    for (int i = 0; i < BI; ++i) rb[i] = ld16(ok ? bptr[i] + (size_t)kt * wstride : zp);
  };
  auto sstore = [&](int buf) {
    u32x4* s = smem + buf * STAGE;
#pragma unroll
    for (int i = 0; i < AI; ++i) s[aoff[i]] = ra[i];
#pragma unroll
    for (int i = 0; i < BI; ++i) s[boff[i]] = rb[i];
  };

  // split-K (EPI_PARTIAL): blockIdx.y owns k-tiles [kt0, nkt)
  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min((K + BK - 1) / BK, kt0 + kt_per_split) : (K + BK - 1) / BK;
  gload(kt0);
  sstore(0);
  __syncthreads();

  for (int kt = kt0; kt < nkt; ++kt) {
    const bool more = kt + 1 < nkt;
    if (more) gload(kt + 1);
    const u32x4* s = smem + ((kt - kt0) & 1) * STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 fa[MT], fb[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        int row = wm * WM + i * 16 + li;
        fa[i] = as_bf16x8(s[row * 8 + ((kk * 4 + g) ^ ((row >> 1) & 7))]);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        int row = wn * 64 + j * 16 + li;
        fb[j] = as_bf16x8(s[BM * 8 + row * 8 + ((kk * 4 + g) ^ ((row >> 1) & 7))]);
      }
      // swapped operands: D'[n][m] so that a lane owns 4 consecutive n of one row m (8-byte stores)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
    }
    if (more) sstore((kt + 1 - kt0) & 1);
    __syncthreads();
  }

  tile_epilogue<EPI, MT, NT>(acc, m0 + wm * WM, n0 + wn * 64, (n0 + wn * 64) / 2, li, g, bias, residual, ldr, C, ldc, M, N, partial, nullptr);
}

// ------------------------------------------------------------------------------------------------
// tiled GEMM v2: LDS-DMA (global_load_lds, 16 B/lane) into a 3-stage LDS ring, counted vmcnt, raw s_barrier
// ------------------------------------------------------------------------------------------------
// Both operands live in LDS in MFMA FRAGMENT ORDER: a 1-KB sub-tile = (16 rows, 32 k) as [4 g][16 rows][8 k], i.e. exactly
// the 64 lanes' 16-byte operands in lane order.  global_load_lds writes wave-uniform-base + lane*16, so one DMA instruction
// fills one sub-tile, and the fragment read is a linear, conflict-free ds_read_b128 (lane reads slot `lane`).  With packed
// weights the W sub-tile is also contiguous in HBM (one 1-KB burst per instruction); row-major operands (activations, or
// an unpacked W) are gathered as 16 rows x 64 B by the per-lane source addresses.
// Pipeline per k-tile:  wait(tile kt landed, leave tile kt+1 in flight) -> s_barrier -> issue DMA of tile kt+2 into the
// stage that was consumed in iteration kt-1 -> MFMAs of tile kt.   No VGPR staging, no ds_write.
template <int BM, int EPI>
__global__ __launch_bounds__(256) void gemm_glds_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, int ldw,
    const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
    bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n, int w_packed,
    float* __restrict__ partial, int kt_per_split) {
  constexpr int BN = 128, BK = 64, NSTAGE = 3;
  constexpr int WM = BM / 2, MT = WM / 16, NT = 4;
  constexpr int A_SUB = (BM / 16) * 2;          // 1-KB sub-tiles of the A tile (row tiles x 2 k-blocks)
  constexpr int B_SUB = (BN / 16) * 2;
  constexpr int STAGE = (A_SUB + B_SUB) * 64;   // 16-byte units per stage
  constexpr int A_PER_WAVE = A_SUB / 4, B_PER_WAVE = B_SUB / 4;
  constexpr int G = A_PER_WAVE + B_PER_WAVE;    // DMA instructions per wave (= per thread) per k-tile
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];

  const int nblk = tiles_m * tiles_n;
  for (int vb = blockIdx.x; vb < nblk; vb += gridDim.x) {     // one tile per block, or a persistent walk under the grid cap
  int bid = vb;
  {
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  const int tn = bid / tiles_m, tm = bid - tn * tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, g = lane >> 4;
  const int K32 = (K + 31) >> 5;
  const bf16_t* zp = reinterpret_cast<const bf16_t*>(lcc_zero_page) + lane * 8;

  // per-lane source pointers of this wave's sub-tiles at k-block 0 (advanced by kb*kstep per k-block)
  const bf16_t* asrc[A_PER_WAVE];
  const bf16_t* bsrc[B_PER_WAVE];
  int akb[A_PER_WAVE], bkb[B_PER_WAVE];
#pragma unroll
  for (int q = 0; q < A_PER_WAVE; ++q) {
    const int st = wave * A_PER_WAVE + q, rt = st >> 1;
    akb[q] = st & 1;
    asrc[q] = A + (size_t)min(m0 + rt * 16 + li, M - 1) * lda + g * 8;
  }
#pragma unroll
  for (int q = 0; q < B_PER_WAVE; ++q) {
    const int st = wave * B_PER_WAVE + q, rt = st >> 1;
    bkb[q] = st & 1;
    const int row = min(n0 + rt * 16 + li, N - 1);
    bsrc[q] = w_packed ? W + (size_t)(row >> 4) * K32 * 512 + lane * 8 : W + (size_t)row * ldw + g * 8;
  }
  const int bstep = w_packed ? 512 : 32;   // elements per 32-k block

  auto issue = [&](int kt, int stage) {
    u32x4* sbase = dsmem + stage * STAGE;
#pragma unroll
    for (int q = 0; q < A_PER_WAVE; ++q) {
      const int kb = kt * 2 + akb[q];
      const bf16_t* src = (kb * 32 + g * 8 < K) ? asrc[q] + kb * 32 : zp;   // A: K % 8 == 0, chunk inside or outside
      glds16(src, lds_addr(sbase + (wave * A_PER_WAVE + q) * 64));
    }
#pragma unroll
    for (int q = 0; q < B_PER_WAVE; ++q) {
      const int kb = kt * 2 + bkb[q];
      const bool ok = w_packed ? (kb < K32) : (kb * 32 + g * 8 < K);
      const bf16_t* src = ok ? bsrc[q] + (size_t)kb * bstep : zp;
      glds16(src, lds_addr(sbase + (A_SUB + wave * B_PER_WAVE + q) * 64));
    }
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min((K + BK - 1) / BK, kt0 + kt_per_split) : (K + BK - 1) / BK;
  issue(kt0, 0);
  if (kt0 + 1 < nkt) issue(kt0 + 1, 1);

  for (int kt = kt0; kt < nkt; ++kt) {
    // tile kt landed (this wave's pieces); the G DMAs of tile kt+1 may stay in flight across the barrier
    if (kt + 1 < nkt) {
      if (G == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();   // every wave's pieces of tile kt are in LDS; everyone finished reading tile kt-1
    if (kt + 2 < nkt) issue(kt + 2, (kt + 2 - kt0) % NSTAGE);
    const u32x4* s = dsmem + ((kt - kt0) % NSTAGE) * STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 fa[MT], fb[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) fa[i] = as_bf16x8(s[((wm * MT + i) * 2 + kk) * 64 + lane]);
#pragma unroll
      for (int j = 0; j < NT; ++j) fb[j] = as_bf16x8(s[(A_SUB + (wn * NT + j) * 2 + kk) * 64 + lane]);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
    }
  }
  tile_epilogue<EPI, MT, NT>(acc, m0 + wm * WM, n0 + wn * 64, (n0 + wn * 64) / 2, li, g, bias, residual, ldr, C, ldc, M, N, partial, nullptr);
  if (vb + (int)gridDim.x < nblk) __syncthreads();     // the next tile's DMA reuses the stages
  }
}

// The last part of a vision q|k|v tile of 32 columns a wave, NW waves: every wave is done with the stages (dsmem), and its DMA pieces have landed
template <int EPI, int BM, int NW, int MT, int NT>
LCC_DEVICE void vit_tile_end(const f32x4 (&acc)[MT][NT], u32x4* dsmem, int m0, int row0, int nbase, int lane, int wave, const bf16_t* bias, bf16_t* C, int ldc, int M, int N,
                             const VitQkvEpi& vq) {
  const int li = lane & 15, g = lane >> 4;
  if constexpr (EPI == EPI_VIT_V) {
    vit_v_epilogue<MT, NT>(acc, m0 + row0, nbase, li, g, bias, M, N, vq);
  } else {
    // cos / sin rows of this tile (gemm_walk_body): clamped reads past the last row belong to rows that are never stored
    constexpr int UNITS = BM * 10;
    const long first = (long)m0 * 10, last = (long)M * 10 - 1;
    for (int t = wave; t * 64 < UNITS; t += NW) {
      const long u = min(first + t * 64 + lane, last);
      glds16(vq.cs + u * 4, lds_addr(dsmem + t * 64));
      glds16(vq.sn + u * 4, lds_addr(dsmem + UNITS + t * 64));
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const float* lcs = reinterpret_cast<const float*>(dsmem);
    vit_qk_epilogue<MT, NT>(acc, m0 + row0, nbase, row0, li, g, bias, C, ldc, M, N, vq.E, lcs, lcs + UNITS * 4);
  }
}

// ------------------------------------------------------------------------------------------------
// 128 x 128 x 64 tile on EIGHT waves with a four-stage LDS-DMA ring: shapes whose 256-column tiles leave most of the chip idle
// ------------------------------------------------------------------------------------------------
// The time is the chain of K / 64 steps of one block, and a split of K would give another summation order.
//   * three stages (96 KB) are in flight;
//   * the fragments of tile kt + 1 are read into a second register set under the MFMAs of tile kt, behind the same barrier;
//   * eight waves, each 64 rows x 32 columns.
// What bounds it: LDS (a step reads 96 KB of fragments and takes 32 KB from the DMA = 1,024 clocks at 128 B/clk against 512 of MFMA per SIMD) and lines
// from beyond the L2 (gemm_strip_kernel).  Same summation order as every other tile kernel of this file.  Measured (us, the tile chosen before -> here): 1000 x 3584,
// K 22528 285 -> 196; 2000 x 1280, K 5120 55 -> 41.
// Requires packed W, K % 64 == 0.  W8: fp8 weights in their packed order, 1 KB a fragment's 64 k, converted in registers in front of the
// MFMAs (the form before wrote the whole weight as bf16 first): 600 x 4608, K 3584 50 -> 34.
constexpr int MID_STAGES = 4;
template <int EPI, bool W8>
LCC_DEVICE void gemm_mid_tile(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual,
    int ldr, bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tm, int tn, float* __restrict__ partial, int kt_per_split,
    const float* __restrict__ wscale, const VitQkvEpi& vq) {
  constexpr int BM = 128, BN = 128, BK = 64, MT = BM / 32, NT = 2, NST = MID_STAGES;
  constexpr int WF = W8 ? 1 : 2;                                  // 1-KB weight sub-tiles of a fragment row
  constexpr int A_UNITS = BM * 8, STAGE = A_UNITS + 8 * WF * 64;  // 16-byte units: [BM rows][8 chunks] (XOR-swizzled) + 16 weight sub-tiles = 32 KB (fp8 weights: 24)
  constexpr int APW = BM / 64, P = APW + WF;                      // DMA pieces of a wave per k-tile: 8 activation rows each, then the weights
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];

  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int li = lane & 15, g = lane >> 4;
  const int K32 = K >> 5, nfrag = (N + 15) >> 4;

  // this wave's DMA pieces of a k-tile: 8 activation rows each, and both 32-k blocks of weight fragment row `wave`
  const bf16_t* asrc[APW];
#pragma unroll
  for (int q = 0; q < APW; ++q) asrc[q] = A + (size_t)min(m0 + (wave + 8 * q) * 8 + (lane >> 3), M - 1) * lda + (((lane & 7) ^ (lane >> 3)) << 3);
  const bf16_t* bsrc = W + (size_t)min((n0 >> 4) + wave, nfrag - 1) * (W8 ? K32 >> 1 : K32) * 512 + lane * 8;
  const unsigned lds0 = lds_addr(dsmem);
  const int nkt_all = K / BK;
  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min(nkt_all, kt0 + kt_per_split) : nkt_all;
  auto issue = [&](int kt, int stage) {           // past the last tile: the source is clamped, the copy lands in a stage nobody reads any more
    const int k = min(kt, nkt - 1);
    const unsigned base = lds0 + (unsigned)(stage * STAGE) * 16u;
#pragma unroll
    for (int q = 0; q < APW; ++q) glds16(asrc[q] + (size_t)k * BK, base + (wave + 8 * q) * 1024u);
#pragma unroll
    for (int h = 0; h < WF; ++h) glds16(bsrc + (size_t)k * (WF * 512) + h * 512, base + (A_UNITS + (wave * WF + h) * 64) * 16u);
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int aoff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) aoff[kk] = (wm * (BM / 2) + li) * 8 + ((W8 ? g * 2 + kk : kk * 4 + g) ^ (li & 7));
  const int boff = A_UNITS + wn * NT * WF * 64 + lane;
  struct Frag { bf16x8 a[2][MT]; u32x4 b[WF][NT]; };
  auto read = [&](Frag& f, int stage) {
    const u32x4* s = dsmem + stage * STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int i = 0; i < MT; ++i) f.a[kk][i] = as_bf16x8(s[aoff[kk] + i * 128]);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if (kk < WF) f.b[kk % WF][j] = s[boff + (j * WF + kk) * 64];
    }
  };
  auto mul = [&](const Frag& f) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 b[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) b[j] = W8 ? fp8x8_to_bf16x8(f.b[0][j][2 * kk], f.b[0][j][2 * kk + 1]) : as_bf16x8(f.b[kk % WF][j]);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = EPI == EPI_VIT_V ? mfma16(f.a[kk][i], b[j], acc[i][j]) : mfma16(b[j], f.a[kk][i], acc[i][j]);
    }
  };
  // tile kt + 1 has landed (this wave's pieces; NST - 3 newer tiles may stay in flight) -> barrier -> DMA of tile kt + NST - 1 into the stage
  // of tile kt - 1 (its fragments were in registers before the barrier) -> fragment reads of tile kt + 1 -> MFMAs of tile kt
  auto step = [&](const Frag& cur, Frag& nxt, int kt, int st) {          // st = stage of tile kt
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * (NST - 3)) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);          // pinned: left alone, hipcc moves the MFMAs of tile kt + 1 up behind its reads
    read(nxt, st == NST - 1 ? 0 : st + 1);
    __builtin_amdgcn_sched_barrier(0);
    issue(kt + NST - 1, st == 0 ? NST - 1 : st - 1);
    mul(cur);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int p = 0; p < NST - 1; ++p) issue(kt0 + p, p);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * (NST - 2)) : "memory");
  __builtin_amdgcn_s_barrier();
  Frag f0, f1;
  read(f0, 0);
  int st = 0, kt = kt0;
  for (; kt + 1 < nkt; kt += 2) {
    step(f0, f1, kt, st);
    st = st == NST - 1 ? 0 : st + 1;
    step(f1, f0, kt + 1, st);
    st = st == NST - 1 ? 0 : st + 1;
  }
  if (kt < nkt) mul(f0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the clamped copies
  if constexpr (EPI == EPI_VIT_QK || EPI == EPI_VIT_V) {
    __builtin_amdgcn_s_barrier();
    vit_tile_end<EPI, BM, 8, MT, NT>(acc, dsmem, m0, wm * (BM / 2), n0 + wn * 32, lane, wave, bias, C, ldc, M, N, vq);
  } else if (wide_rows<EPI>(C, ldc, bias, residual, ldr)) {
    __builtin_amdgcn_s_barrier();          // every wave is done with the stages, and its DMA pieces have landed
    tile_epilogue_wide<EPI, MT, NT>(acc, m0 + wm * (BM / 2), n0 + wn * 32, lane, bias, residual, ldr, C, ldc, M, N, wscale,
                                    reinterpret_cast<unsigned char*>(dsmem) + wave * 4096);
  } else tile_epilogue<EPI, MT, NT>(acc, m0 + wm * (BM / 2), n0 + wn * 32, (n0 + wn * 32) / 2, li, g, bias, residual, ldr, C, ldc, M, N, partial, wscale);
}
template <int EPI, bool W8>
__global__ __launch_bounds__(512) void gemm_mid_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual,
    int ldr, bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n, float* __restrict__ partial, int kt_per_split,
    const float* __restrict__ wscale, int raster, VitQkvEpi vq) {
  const int nblk = tiles_m * tiles_n;
  for (int vb = blockIdx.x; vb < nblk; vb += gridDim.x) {     // one tile per block, or a persistent walk under the grid cap
  int bid = vb;
  {
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  int tn, tm;                                     // tile order: see gemm_big_kernel
  if (raster > 0) {
    const int band = bid / (raster * tiles_m), rem = bid - band * raster * tiles_m;
    const int bw = min(raster, tiles_n - band * raster);
    tm = rem / bw;
    tn = band * raster + (rem - tm * bw);
  } else {
    tn = bid / tiles_m;
    tm = bid - tn * tiles_m;
  }
  if constexpr (EPI == EPI_VIT_QKV) {
    const int qk_tiles = 2 * vq.E / 128;          // V: rows 2E.. of the packed weight
    if (tn >= qk_tiles)
      gemm_mid_tile<EPI_VIT_V, W8>(A, lda, W + (size_t)2 * vq.E * K, bias != nullptr ? bias + 2 * vq.E : nullptr, nullptr, 0, nullptr, 0, M, vq.E, K, tm, tn - qk_tiles, nullptr, 0, nullptr, vq);
    else gemm_mid_tile<EPI_VIT_QK, W8>(A, lda, W, bias, nullptr, 0, C, ldc, M, 2 * vq.E, K, tm, tn, nullptr, 0, nullptr, vq);
  } else gemm_mid_tile<EPI, W8>(A, lda, W, bias, residual, ldr, C, ldc, M, N, K, tm, tn, partial, kt_per_split, wscale, vq);
  if (vb + (int)gridDim.x < nblk) __syncthreads();     // the next tile's DMA reuses the stages
  }
}

// ------------------------------------------------------------------------------------------------
// The 64 x 128 tile: FOUR waves, one a SIMD, each 64 rows x 32 columns; the weights go from memory into registers
// ------------------------------------------------------------------------------------------------
// With 32 columns of its own a wave is the only reader of its weight fragments: LDS holds the activations alone, and a k-step moves 32 + 8 KB through it instead
// of 64 + 24 (gemm_mid_kernel's form: 32 x 32 a wave).  One step in source order: the activation fragments of tile kt + 1, a piece of what tile kt + D - 1 needs
// and the MFMAs of tile kt by turns, so that a wave alone on its SIMD is never held by a burst of loads.
// What bounds it then: what a compute unit takes from beyond its L2.  Lines that are there arrive at 135-150 B/ns, lines that the blocks of an XCD ask for
// together and that come from memory at 45-58, whatever is in flight (2 to 8 steps measured the same): 24 KB a step are 0.16 us or 0.42.  So
//   * compute units that get no tile read the weight ahead of the others into the memory-side cache (strip_fetch), whose lines come sooner than DRAM's;
//   * nothing is requested past the last tile but what the full groups of D steps do.
// Measured (us, weights from memory; the eight-wave form before -> these -> with fetching blocks): 1456 x 1280, K 5120 35.3 -> 33.0 -> 28.1, K 1280 10.6 -> 9.8;
// 720 x 1280, K 5120 29.2 -> 28.7 -> 25.4; 390 x 3584, K 3584 23.7 -> 22.4 -> 20.6; 1120 x 1280, K 5184 30.9 -> 30.3 -> 25.1.
// Not taken: weight loads past the caches (nt: 33 -> 40, the other blocks of the XCD fetch them again), 8 to 12 steps ahead (no faster), a dword of every line ahead of
// its use by the block itself (loads return in order: slower), 128 rows x 32 columns a wave (2 to 4 % either way of gemm_mid_kernel).
// Same summation order as every other tile kernel of this file.  Requires packed W, K % 64 == 0.  W8: fp8 weights in their packed order, 1 KB a fragment's 64 k,
// converted in registers in front of the MFMAs.
// Blocks without a tile read 2 KB of every fragment row by turns, from piece c0 to c1 of the rows (`row` pieces of 16 bytes each), in the order in which the others will
LCC_DEVICE void strip_fetch(const bf16_t* W, int row, int nfrag, int c0, int c1, int e, int ne) {
  const u32x4* src = reinterpret_cast<const u32x4*>(W) + (threadIdx.x & 127);
  const int half = threadIdx.x >> 7, pairs = (nfrag + 1) >> 1, items = (c1 - c0) * pairs;
  for (int i0 = e; i0 < items; i0 += 8 * ne) {
    u32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = min(i0 + u * ne, items - 1), c = i / pairs, fr = min((i - c * pairs) * 2 + half, nfrag - 1);
      v[u] = src[(size_t)fr * row + (size_t)(c0 + c) * 128];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) asm volatile("" ::"v"(v[u]));
  }
}
template <int... U, class F>
LCC_DEVICE void strip_steps(std::integer_sequence<int, U...>, F f) { (f(std::integral_constant<int, U>{}), ...); }
template <int EPI, bool W8>
LCC_DEVICE void gemm_strip_tile(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual,
    int ldr, bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tm, int tn, float* __restrict__ partial, int kt_per_split,
    const float* __restrict__ wscale, const VitQkvEpi& vq) {
  constexpr int BM = 64, BK = 64, MT = BM / 16, NT = 2, D = STRIP_STAGES;
  constexpr int WF = W8 ? 1 : 2;                                  // 1-KB weight sub-tiles of a fragment row
  constexpr int STAGE = BM * 8;                                   // 16-byte units: [BM rows][8 chunks] (XOR-swizzled) = 8 KB
  constexpr int APW = BM / 32, P = APW + WF * NT;                 // a wave's memory instructions of a k-tile: 8 activation rows each, then its weights
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];
  static_assert((D & 1) == 0 && P <= 2 * MT, "the two fragment sets alternate; a piece beside every fragment");

  const int nkt_all = K / BK;
  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min(nkt_all, kt0 + kt_per_split) : nkt_all;
  const int m0 = tm * BM, n0 = tn * 128;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int nfrag = (N + 15) >> 4;

  const bf16_t* asrc[APW];
#pragma unroll
  for (int q = 0; q < APW; ++q) asrc[q] = A + (size_t)min(m0 + (wave + 4 * q) * 8 + (lane >> 3), M - 1) * lda + (((lane & 7) ^ (lane >> 3)) << 3);
  const bf16_t* bsrc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) bsrc[j] = W + (size_t)min((n0 >> 4) + wave * NT + j, nfrag - 1) * (nkt_all * WF) * 512 + lane * 8;
  const unsigned lds0 = lds_addr(dsmem) + wave * 1024u;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int aoff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) aoff[kk] = li * 8 + ((W8 ? g * 2 + kk : kk * 4 + g) ^ (li & 7));
  bf16x8 f[2][2][MT];                             // activation fragments of two k-tiles
  u32x4 w[D][WF][NT];                             // weights of D
  // piece q of k-tile k (in range) into stage and weight set u
  auto issue = [&](int q, int k, auto uc) {
    constexpr int u = decltype(uc)::value;
    if (q < APW) glds16(asrc[q < APW ? q : 0] + (size_t)k * BK, lds0 + (unsigned)(u * STAGE * 16 + (q < APW ? q : 0) * 4096));
    else if (q < P) {
      const int h = (q - APW) / NT, j = (q - APW) % NT;
      w[u][h % WF][j] = ld16(bsrc[j] + (size_t)k * (WF * 512) + h * 512);
    }
  };
  // The stage and weight set of tile kt is u.  Tile kt + 1 has landed (the waits count every piece issued behind it: the barriers to the scheduler keep them in this
  // order) -> block barrier -> its fragments are read, tile kt + D - 1 goes into the stage and the registers of tile kt - 1, whose fragments were in registers before
  // the barrier, and tile kt is multiplied.  DRAIN > 0: the last steps, with nothing to request (past the last tile sources are clamped: stages nobody reads any more)
  auto step = [&](int kt, auto uc, auto dc) {
    constexpr int u = decltype(uc)::value, drain = decltype(dc)::value;
    constexpr std::integral_constant<int, (u + D - 1) % D> un{};
    const int k = min(kt + D - 1, nkt - 1);
    const u32x4* s = dsmem + ((u + 1) % D) * STAGE;
    constexpr int behind = drain == 0 ? D - 3 : D - 2 - drain;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(behind > 0 ? P * behind : 0) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 b[2][NT];
#pragma unroll
    for (int q = 0; q < 2 * MT; ++q) {
      const int kk = q / MT, i = q % MT;
      f[(u + 1) & 1][kk][i] = as_bf16x8(s[aoff[kk] + i * 128]);
      if (drain == 0) issue(q, k, un);
      if (i == 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) b[kk][j] = W8 ? fp8x8_to_bf16x8(w[u][0][j][2 * kk], w[u][0][j][2 * kk + 1]) : as_bf16x8(w[u][kk % WF][j]);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = EPI == EPI_VIT_V ? mfma16(f[u & 1][kk][i], b[kk][j], acc[i][j]) : mfma16(b[kk][j], f[u & 1][kk][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  __builtin_amdgcn_sched_barrier(0);
  strip_steps(std::make_integer_sequence<int, D - 1>{}, [&](auto uc) {
#pragma unroll
    for (int q = 0; q < P; ++q) issue(q, min(kt0 + decltype(uc)::value, nkt - 1), uc);
    __builtin_amdgcn_sched_barrier(0);
  });
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * (D - 2)) : "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < 2 * MT; ++q) f[0][q / MT][q % MT] = as_bf16x8(dsmem[aoff[q / MT] + (q % MT) * 128]);
  int kt = kt0;
  for (; kt + D <= nkt; kt += D) strip_steps(std::make_integer_sequence<int, D>{}, [&](auto uc) { step(kt + decltype(uc)::value, uc, std::integral_constant<int, 0>{}); });
  const int rem = nkt - kt;
  strip_steps(std::make_integer_sequence<int, D - 1>{}, [&](auto uc) {
    if (decltype(uc)::value < rem) step(kt + decltype(uc)::value, uc, std::integral_constant<int, decltype(uc)::value + 1>{});
  });
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the clamped copies
  if constexpr (EPI == EPI_VIT_QK || EPI == EPI_VIT_V) {
    __builtin_amdgcn_s_barrier();
    vit_tile_end<EPI, BM, 4, MT, NT>(acc, dsmem, m0, 0, n0 + wave * 32, lane, wave, bias, C, ldc, M, N, vq);
  } else if (wide_rows<EPI>(C, ldc, bias, residual, ldr)) {
    __builtin_amdgcn_s_barrier();          // every wave is done with the stages, and its DMA pieces have landed
    tile_epilogue_wide<EPI, MT, NT>(acc, m0, n0 + wave * 32, lane, bias, residual, ldr, C, ldc, M, N, wscale,
                                    reinterpret_cast<unsigned char*>(dsmem) + wave * 4096);
  } else tile_epilogue<EPI, MT, NT>(acc, m0, n0 + wave * 32, (n0 + wave * 32) / 2, li, g, bias, residual, ldr, C, ldc, M, N, partial, wscale);
}
template <int EPI, bool W8>
__global__ __launch_bounds__(256, 2) void gemm_strip_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual,
    int ldr, bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n, float* __restrict__ partial, int kt_per_split,
    const float* __restrict__ wscale, int raster, int fetch, VitQkvEpi vq) {
  constexpr int WF = W8 ? 1 : 2;
  const int nkt_all = K / 64;
  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min(nkt_all, kt0 + kt_per_split) : nkt_all;
  const int nblk = tiles_m * tiles_n;
  if ((int)blockIdx.x >= nblk) {                  // the last `fetch` k-tiles of this split
    strip_fetch(W, nkt_all * WF * 64, (N + 15) >> 4, max(kt0, nkt - fetch) * WF / 2, nkt * WF / 2, (int)blockIdx.x - nblk, (int)gridDim.x - nblk);
    return;
  }
  for (int vb = blockIdx.x; vb < nblk; vb += gridDim.x) {     // one tile per block, or a persistent walk under the grid cap
  int bid = vb;
  {
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  int tn, tm;                                     // tile order: see gemm_big_kernel
  if (raster > 0) {
    const int band = bid / (raster * tiles_m), rem = bid - band * raster * tiles_m;
    const int bw = min(raster, tiles_n - band * raster);
    tm = rem / bw;
    tn = band * raster + (rem - tm * bw);
  } else {
    tn = bid / tiles_m;
    tm = bid - tn * tiles_m;
  }
  if constexpr (EPI == EPI_VIT_QKV) {
    const int qk_tiles = 2 * vq.E / 128;          // V: rows 2E.. of the packed weight
    if (tn >= qk_tiles)
      gemm_strip_tile<EPI_VIT_V, W8>(A, lda, W + (size_t)2 * vq.E * K, bias != nullptr ? bias + 2 * vq.E : nullptr, nullptr, 0, nullptr, 0, M, vq.E, K, tm, tn - qk_tiles, nullptr, 0, nullptr, vq);
    else gemm_strip_tile<EPI_VIT_QK, W8>(A, lda, W, bias, nullptr, 0, C, ldc, M, 2 * vq.E, K, tm, tn, nullptr, 0, nullptr, vq);
  } else gemm_strip_tile<EPI, W8>(A, lda, W, bias, residual, ldr, C, ldc, M, N, K, tm, tn, partial, kt_per_split, wscale, vq);
  if (vb + (int)gridDim.x < nblk) __syncthreads();     // the next tile's DMA reuses the stages
  }
}

// ------------------------------------------------------------------------------------------------
// tiled GEMM v3: 8 waves, BM x 256 x 64 block tile (BM = 256 or 128), LDS-DMA for both operands
// ------------------------------------------------------------------------------------------------
// The 64x128 / 128x128 tiles above move (1/BM + 1/BN) bytes per flop from L2 into LDS = 0.023 / 0.016 B/flop, i.e. 95 / 64
// B/clk/CU at the MFMA peak -- above what the L2->CU path delivers, so they top out at 20-29 % of the bf16 peak.  A 256x256
// tile needs 0.0078 B/flop (32 B/clk/CU).  8 waves = 2 (M) x 4 (N), wave tile (BM/2) x 64, 64 MFMAs per wave per k-tile.
//   * W (packed fragment order in HBM): one DMA instruction copies one 1-KB (16 rows, 32 k) fragment sub-tile; the fragment
//     read is the linear, conflict-free ds_read_b128 of slot `lane` (as in gemm_glds_kernel).
//   * A (row-major activations): staged in FULL 128-byte lines -- one DMA instruction = 8 rows x 128 B -- into a [BM][8 x 16 B]
//     image whose 16-byte chunks are XOR-swizzled with (row & 7).  LDS-DMA writes lane-linear, so the swizzle is applied to
//     the per-lane SOURCE chunk and again on the fragment read (the same involution on both sides).  Full-line reads keep the
//     texture-address path at one request per 128 B instead of the 16 rows x 64 B gather of a fragment-shaped load.
//   * pipeline: BM = 256: two 64-KB stages (128 KB), vmcnt(0) + s_barrier per k-tile, the DMA of tile kt+1 runs under the
//     MFMAs of tile kt.  BM = 128: three 48-KB stages, counted vmcnt so that one tile stays in flight across the barrier.
// Requires packed W, K % 64 == 0 (every shape of the 7B/2B/72B models except the 1176-wide patch embedding).
// W8 = true: W is fp8 e4m3 in the PACKED8 order (one 1-KB DMA = a 16-row x 64-k fragment = both k-steps of a k-tile); the
// fragment read is one ds_read_b128 per 16 rows whose halves are converted to bf16 in registers, and the activation chunk
// order follows PACKED8's k assignment (MFMA h of lane group g takes k = g*16 + h*8 ..).  Half the W bytes in L2 and LDS;
// the stage shrinks to 48 KB (BM 256) so that three stages fit and one tile stays in flight across the barrier.
// (the kernel proper is gemm_big_kernel below: it maps blockIdx to a tile (tm, tn) and runs this body)
template <int BM, int EPI, int SCHED, bool W8>
LCC_DEVICE void gemm_big_body(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
    const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
    bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tm, int tn,
    float* __restrict__ partial, int kt_per_split, const float* __restrict__ wscale) {
  constexpr int BN = 256, BK = 64, NSTAGE = (BM >= 192 && !W8) ? 2 : 3;     // BM 192 (round 4): 56-KB stages, two of them
  constexpr int WM = BM / 2, MT = WM / 16, NT = 4;
  constexpr int A_UNITS = BM * 8;                 // 16-byte units of the A image
  constexpr int B_SUB = (BN / 16) * (W8 ? 1 : 2); // 1-KB fragment sub-tiles of the W tile
  constexpr int STAGE = A_UNITS + B_SUB * 64;     // 16-byte units per stage
  constexpr int A_PER_WAVE = BM / 64;             // 8-row x 128-B pieces per wave (BM/8 pieces over 8 waves)
  constexpr int B_PER_WAVE = B_SUB / 8;
  constexpr int G = A_PER_WAVE + B_PER_WAVE;      // DMA instructions per wave per k-tile
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];

  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int li = lane & 15, g = lane >> 4;
  const int K32 = K >> 5, nfrag = N >> 4;
  const bool wave_has_rows = m0 + wm * WM < M;

  const bf16_t* asrc[A_PER_WAVE];
  const bf16_t* bsrc[B_PER_WAVE];
#pragma unroll
  for (int q = 0; q < A_PER_WAVE; ++q) {
    const int row = (wave * A_PER_WAVE + q) * 8 + (lane >> 3);
    asrc[q] = A + (size_t)min(m0 + row, M - 1) * lda + (((lane & 7) ^ (lane >> 3)) << 3);
  }
#pragma unroll
  for (int q = 0; q < B_PER_WAVE; ++q) {
    const int st = wave * B_PER_WAVE + q;
    if (W8) {                                      // sub-tile = n-fragment row st, all 64 k of the tile (1 KB of fp8)
      const int fr = min((n0 >> 4) + st, nfrag - 1);
      bsrc[q] = W + ((size_t)fr * (K >> 6)) * 512 + lane * 8;          // bf16_t units: 1024 B = 512 units per fragment
    } else {                                       // sub-tile: n-fragment row st >> 1, 32-k block st & 1
      const int fr = min((n0 >> 4) + (st >> 1), nfrag - 1);
      bsrc[q] = W + ((size_t)fr * K32 + (st & 1)) * 512 + lane * 8;
    }
  }

  auto issue = [&](int kt, int stage) {
    u32x4* sbase = dsmem + stage * STAGE;
#pragma unroll
    for (int q = 0; q < A_PER_WAVE; ++q)
      glds16((asrc[q] + kt * BK), lds_addr(sbase + (wave * A_PER_WAVE + q) * 64));
#pragma unroll
    for (int q = 0; q < B_PER_WAVE; ++q)
      glds16((bsrc[q] + (size_t)kt * (W8 ? 512 : 1024)), lds_addr(sbase + A_UNITS + (wave * B_PER_WAVE + q) * 64));
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int nkt_all = K / BK;
  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min(nkt_all, kt0 + kt_per_split) : nkt_all;
#pragma unroll
  for (int p = 0; p < NSTAGE - 1; ++p)
    if (kt0 + p < nkt) issue(kt0 + p, p);

  // fragment read offsets (16-byte units within a stage)
  int aoff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) aoff[kk] = (wm * WM + li) * 8 + ((W8 ? g * 2 + kk : kk * 4 + g) ^ (li & 7));
  const int boff = A_UNITS + (wn * NT * (W8 ? 1 : 2)) * 64 + lane;

  for (int kt = kt0; kt < nkt; ++kt) {
    // this wave's pieces of tile kt have landed; NSTAGE-2 later tiles may stay in flight across the barrier
    if (NSTAGE == 3 && kt + 1 < nkt) {
      if (G == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else if (G == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();   // tile kt complete in LDS; every wave is done reading tile kt-1
    // SCHED 6 issues the same pieces one at a time between the row tiles of MFMAs below (a burst of 8 DMA instructions right after the
    // barrier holds the wave's issue port for ~60-100 cycles each while BOTH waves of the SIMD are at the same point)
    if (SCHED != 6 && kt + NSTAGE - 1 < nkt) issue(kt + NSTAGE - 1, (kt + NSTAGE - 1 - kt0) % NSTAGE);
    const u32x4* s = dsmem + ((kt - kt0) % NSTAGE) * STAGE;
    // ragged last row tile (e.g. M = 386 = 3 x 128 + 2): a wave whose WM rows are all past M skips the multiply and only keeps
    // feeding the DMA ring and the barriers (wave-uniform branch around the whole k-tile body; a finer per-16-row predicate
    // made hipcc if-convert the accumulators and spill)
    if (!wave_has_rows) {
      if (SCHED == 6 && kt + NSTAGE - 1 < nkt) issue(kt + NSTAGE - 1, (kt + NSTAGE - 1 - kt0) % NSTAGE);   // no MFMA stream to spread them over
    } else if (SCHED == 0) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        bf16x8 fa[MT], fb[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if (W8) { const u32x4 raw = s[boff + j * 64]; fb[j] = fp8x8_to_bf16x8(raw[2 * kk], raw[2 * kk + 1]); }
          else fb[j] = as_bf16x8(s[boff + (j * 2 + kk) * 64]);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) fa[i] = as_bf16x8(s[aoff[kk] + i * 128]);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
      }
    } else {
      // explicit software pipeline of the fragment reads: the 8 W fragments of the k-tile are read up front, the activation
      // fragments stream through a 3-register ring two steps (8 MFMAs = 128 cycles) ahead of their use; the issue order is
      // pinned with sched_group_barrier (DS read = 0x100, MFMA = 0x008) so that hipcc does not fall back to read-wait-use.
      bf16x8 fb[2][NT], fa[3];
      if (W8) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const u32x4 raw = s[boff + j * 64];
          fb[0][j] = fp8x8_to_bf16x8(raw[0], raw[1]);
          fb[1][j] = fp8x8_to_bf16x8(raw[2], raw[3]);
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int j = 0; j < NT; ++j) fb[kk][j] = as_bf16x8(s[boff + (j * 2 + kk) * 64]);
      }
      fa[0] = as_bf16x8(s[aoff[0]]);
      fa[1] = as_bf16x8(s[aoff[0] + 128]);
      // SCHED 6: piece t of the NEXT ring tile goes out after row-tile step t.  Unconditional (a branch would cut the scheduling
      // region): past the last tile the source is clamped and the copy lands in a stage nobody reads any more.
      const int kt_dma = min(kt + NSTAGE - 1, nkt - 1);
      u32x4* dma_base = dsmem + ((kt + NSTAGE - 1 - kt0) % NSTAGE) * STAGE;
#pragma unroll
      for (int t = 0; t < 2 * MT; ++t) {
        if (t + 2 < 2 * MT) fa[(t + 2) % 3] = as_bf16x8(s[aoff[(t + 2) / MT] + ((t + 2) % MT) * 128]);
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[t % MT][j] = mfma16(fb[t / MT][j], fa[t % 3], acc[t % MT][j]);
        if (SCHED == 6 && t < G) {
          if (t < A_PER_WAVE)
            glds16((asrc[t < A_PER_WAVE ? t : 0] + kt_dma * BK), lds_addr(dma_base + (wave * A_PER_WAVE + t) * 64));
          else
            glds16((bsrc[t >= A_PER_WAVE ? t - A_PER_WAVE : 0] + (size_t)kt_dma * (W8 ? 512 : 1024)), lds_addr(dma_base + A_UNITS + (wave * B_PER_WAVE + (t - A_PER_WAVE)) * 64));
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x100, (W8 ? NT : 2 * NT) + 2, 0);
#pragma unroll
      for (int t = 0; t < 2 * MT; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
        if (SCHED == 6 && t < G) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);      // one VMEM (the LDS-DMA piece)
      }
    }
  }
  if (SCHED == 6) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the clamped copies of the last iterations
  if constexpr (EPI == EPI_PARTIAL) {
    __builtin_amdgcn_s_barrier();          // every wave is done with the stages, and its DMA pieces have landed
    tile_slab_wide<MT, NT>(acc, m0 + wm * WM, n0 + wn * 64, lane, M, N, partial, wscale, reinterpret_cast<unsigned char*>(dsmem) + wave * 8192);
  } else if (wide_rows<EPI>(C, ldc, bias, residual, ldr)) {
    __builtin_amdgcn_s_barrier();          // every wave is done with the stages, and its DMA pieces have landed
    tile_epilogue_wide<EPI, MT, NT>(acc, m0 + wm * WM, n0 + wn * 64, lane, bias, residual, ldr, C, ldc, M, N, wscale,
                                    reinterpret_cast<unsigned char*>(dsmem) + wave * 8192);
  } else tile_epilogue<EPI, MT, NT>(acc, m0 + wm * WM, n0 + wn * 64, (n0 + wn * 64) / 2, li, g, bias, residual, ldr, C, ldc, M, N, partial, wscale);
}

template <int BM, int EPI, int SCHED, bool W8>
__global__ __launch_bounds__(512) void gemm_big_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
    const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
    bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n,
    float* __restrict__ partial, int kt_per_split, const float* __restrict__ wscale, int raster) {
  const int nblk = tiles_m * tiles_n;
  for (int vb = blockIdx.x; vb < nblk; vb += gridDim.x) {     // one tile per block, or a persistent walk under the grid cap
  int bid = vb;
  {
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  // tile id -> (tm, tn).  An XCD (one L2) runs a contiguous range of ids, ~32 of them at a time.
  //   raster 0: column-major -- the 32 share ~2.5 W panels and ALL row panels (M = 3088: 13 + 2.5 panels of 1.8 MB per 32 tiles);
  //   raster G (round 5): bands of G column tiles, row-major inside a band -- 32 consecutive ids are a (32 / G) x G super-tile
  //   (G = 8: 4 + 8 panels per 32 tiles: 0.77 x the bytes from beyond the L2, and the four blocks of a W panel run side by side).
  int tn, tm;
  if (raster > 0) {
    const int band = bid / (raster * tiles_m), rem = bid - band * raster * tiles_m;
    const int bw = min(raster, tiles_n - band * raster);       // the last band may be narrower
    tm = rem / bw;
    tn = band * raster + (rem - tm * bw);
  } else {
    tn = bid / tiles_m;
    tm = bid - tn * tiles_m;
  }
  gemm_big_body<BM, EPI, SCHED, W8>(A, lda, W, bias, residual, ldr, C, ldc, M, N, K, tm, tn, partial, kt_per_split, wscale);
  if (vb + (int)gridDim.x < nblk) __syncthreads();     // the next tile's DMA reuses the stages
  }
}

// ------------------------------------------------------------------------------------------------
// the same tiles, walked: one block a compute unit goes through its tiles with the DMA ring running on from tile to tile, and the two waves of a SIMD
// take turns at its matrix pipe
// ------------------------------------------------------------------------------------------------
// Turns.  Waves w and w + 4 share a SIMD.  A k-tile of a wave is two phases -- the first half of its row fragments, then the second -- and a phase two slots
// with a barrier behind each: in the first the wave reads the phase's fragments and issues DMA pieces, in the second it multiplies.  Waves 4..7 are one slot
// behind, so that one wave of a SIMD multiplies (32 MFMAs back to back at 256 rows, operands all in registers) while the other reads: with both in step
// (before: reads between the MFMAs of either, one barrier a k-tile) the matrix pipe waited for LDS and barriers a quarter of the time.
// A row of launches on weights from memory, us, in step -> here: 4096 x 3584, K 18944 460 -> 390; 4096 x 18944, K 3584 460 -> 420; 8192-cube 800 -> 728
// (1.51 PF; the MFMAs alone, on such data, hold 1.755 GHz = 1.85 PF).  Tried there: s_setprio around the MFMAs 1-4 % slower; the pieces between the MFMAs
// instead of behind the reads 437 (K 18944); phases by k halves, which balance the reads but free a stage late, 460.
//
// Ring.  Stage = [rows][8 x 16 B] activations (XOR-swizzled) + 32 weight sub-tiles.  What phase 0 reads (first halves of the rows, all weights) is filled
// again in the next phase 1, what phase 1 reads (second halves) in the next phase 0: two slots later, when either wave's reads are back.  A phase's rows of a
// stage are the same for tiles of every height (ROW1), so that this holds from a tile to a taller one too.  Pieces leave in the order
// in which they are needed, so "all but the last (NSTAGE - 1) k-tiles' worth have landed" is the wait of every phase.  They run on into the
// next tile, whose first stages land while this one's results leave through LDS of their own; stores drain under the next tile's first phases (vmcnt retires
// in order: a wait counts the pieces and lets the younger stores be, if all of them were issued -- inner tiles).
// The first wave of a SIMD stores its results while the second is still multiplying, and the second in the slot in which the first begins the next tile.
//
// Rows: 256, 192, 160 or 128 (BM), or VARIABLE (BM 272): 16, 17 or 18 row fragments a tile.  M is whatever the turn packs: 8 co-scheduled streaming chunks are 8 x 386 =
// 3088 rows = 12 x 256 + 16, so a 13th row tile of 256 would multiply 16 live rows and 13 x 148 = 1924 blocks be 7.5 rounds of the 256 CUs.  The F = ceil(M / 16)
// fragments are dealt out over F / 18 to F / 16 tiles (vh_tiles), the first F % tiles of them one fragment taller (3088 rows: 11 tiles of 256 + one of 272 = 6.94 rounds;
// 3436: 12 of 288 / 272); the two wave rows split f fragments f / 2 : f - f / 2, one copy of the k loop per count.
// A slot without rows (192, 160 and variable rows) copies one 16-byte piece into a scratch: the stream of pieces is the same in every wave.
// Bits as gemm_big_kernel (same k order per output).  fp8 weights (W8) are converted behind the LDS read, beside the other wave's MFMAs; [37888, 3584] with SwiGLU,
// us, in step and 128 or 256 rows -> here: 514 rows 175 -> 145, 772 274 -> 196, 1158 293 -> 265, 1544 447 -> 378, 3088 696 -> 628; [3584, 18944], 2316 rows 384 -> 286.  The vision q|k|v epilogues (gemm_vit_kernel) run a tile a block: their rotation tables need
// the stages (15,840 x 3840, K 1280: 182 -> 172 us).  Grid: at most 256 blocks over all splits (one a compute unit), or the cap.
template <int BM, int EPI, bool W8 = false>
struct Walk {
  static constexpr bool VH = BM == 272;
  static constexpr int ROWS = VH ? 288 : BM, MT = VH ? 8 : BM / 32, MTX = VH ? 9 : MT;             // row fragments of a wave (variable rows: 8 or 9)
  static constexpr int H0 = VH ? 4 : (MT + 1) / 2, H1 = MTX - H0;                                  // of phase 0, at most of phase 1
  static constexpr int P0 = (4 * H0 + 7) / 8, P1 = (4 * H1 + 7) / 8, PB = W8 ? 2 : 4, G = P0 + PB + P1;     // a wave's pieces of a k-tile: rows of phase 0, weights; rows of phase 1
  static constexpr bool SPARE = VH || (4 * H0) % 8 != 0 || (4 * H1) % 8 != 0;                      // slots without rows
  static constexpr int ROW1 = VH ? 16 * MTX : BM / 2;                                              // of the stage: the second wave row's first, whatever a tile's height
  static constexpr int NSTAGE = BM == 128 ? 3 : 2;
  static constexpr int A_UNITS = ROWS * 8, STAGE = A_UNITS + PB * 512;                             // 16-byte units
  static constexpr int EGR = BM >= 160 && !VH && EPI != EPI_GELU_ERF ? 2 : 1;                      // row tiles of an epilogue group: 2 KB of LDS a wave each (the erf: registers)
  static constexpr unsigned SCRATCH = (unsigned)NSTAGE * STAGE * 16u, EPILOGUE = SCRATCH + (SPARE ? 1024u : 0u);
  static constexpr size_t LDS = EPILOGUE + 8 * EGR * 2048;
  static constexpr int LATER = G * (NSTAGE - 1);                                                   // pieces that may be on their way behind those that are read next
  static constexpr int NSTORE = EPI == EPI_PARTIAL ? MT * 4 : MT * 2;                              // stores of a wave in the epilogue of an inner tile
  static_assert(LDS <= 163840, "LDS of a compute unit");
  static_assert(LATER + NSTORE <= 63, "vmcnt");
};
template <int BM, int EPI, bool W8 = false>
LCC_DEVICE void gemm_walk_body(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
    const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
    bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n,
    float* __restrict__ partial, int kt_per_split, int raster, const VitQkvEpi& vq = VitQkvEpi(), int one_m = 0, int one_n = 0,
    const float* __restrict__ wscale = nullptr) {
  using S = Walk<BM, EPI, W8>;
  constexpr bool VIT = EPI == EPI_VIT_QK || EPI == EPI_VIT_V;      // the tile (one_m, one_n) alone: the rotation's tables take the stages
  constexpr int BN = 256, BK = 64, NT = 4, NSTAGE = S::NSTAGE, STAGE = S::STAGE, H0 = S::H0, P0 = S::P0, P1 = S::P1, PB = S::PB, LATER = S::LATER;
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int li = lane & 15, g = lane >> 4;
  const int K32 = K >> 5, nfrag = N >> 4;
  const int nblk = VIT ? 1 : tiles_m * tiles_n, step = VIT ? 1 : gridDim.x, vb0 = VIT ? 0 : blockIdx.x;
  const int F = (M + 15) >> 4, fbase = S::VH ? F / tiles_m : 0, frem = S::VH ? F - fbase * tiles_m : 0;
  const int nkt_all = K / BK;
  const int kt0 = (EPI == EPI_PARTIAL) ? blockIdx.y * kt_per_split : 0;
  const int nkt = (EPI == EPI_PARTIAL) ? min(nkt_all, kt0 + kt_per_split) : nkt_all;

  auto tile_of = [&](int bid, int& m0, int& n0, int& row1, int& rows) {     // tile order: see gemm_big_kernel; row1: the second wave row's first; rows: of the tile
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
    int tn, tm;
    if (VIT) {
      tm = one_m;
      tn = one_n;
    } else if (raster > 0) {
      const int band = bid / (raster * tiles_m), rem = bid - band * raster * tiles_m;
      const int bw = min(raster, tiles_n - band * raster);
      tm = rem / bw;
      tn = band * raster + (rem - tm * bw);
    } else {
      tn = bid / tiles_m;
      tm = bid - tn * tiles_m;
    }
    const int f = S::VH ? __builtin_amdgcn_readfirstlane(fbase + (tm < frem ? 1 : 0)) : BM / 16;
    m0 = __builtin_amdgcn_readfirstlane(S::VH ? (tm * fbase + min(tm, frem)) << 4 : tm * BM);
    n0 = __builtin_amdgcn_readfirstlane(tn * BN);
    row1 = (f >> 1) * 16;
    rows = f * 16;
  };
  // The pieces of phase 0 and of phase 1 each go their own way through (tile, k-tile).  Scalar bases, a 32-bit offset per lane and piece inside the tile.
  // A slot's rows: 8 of the first wave row's part, behind them the second's; none: one 16-byte piece into the scratch
  struct Way { int vb, kt; const bf16_t* a; };
  Way w0 = {vb0, kt0, nullptr}, w1 = w0;
  const bf16_t* bbase[2];
  unsigned off0[P0], off1[P1], dst0[P0], dst1[P1];
  const unsigned swz = ((lane & 7) ^ (lane >> 3)) << 4, row_bytes = (unsigned)(lda * 2);
  auto slot = [&](int p, int from, int n_first, int n_second, int row1, int m0, unsigned& off, unsigned& dst) {
    const int row = p < n_first ? from + p * 8 : p < n_first + n_second ? S::ROW1 + from + (p - n_first) * 8 : -1;          // of the stage
    off = row >= 0 ? (unsigned)min((S::VH && p >= n_first ? row - (S::ROW1 - row1) : row) + (lane >> 3), M - 1 - m0) * row_bytes + swz : 0u;
    dst = row >= 0 ? (unsigned)row * 128u : S::SCRATCH;
  };
  auto point0 = [&] {
    int m0, n0, row1, rows;
    tile_of(w0.vb, m0, n0, row1, rows);
    w0.a = A + (size_t)m0 * lda;
#pragma unroll
    for (int q = 0; q < 2; ++q) bbase[q] = W + (size_t)min((n0 >> 4) + wave * 2 + q, nfrag - 1) * (W8 ? K >> 6 : K32) * 512;
#pragma unroll
    for (int q = 0; q < P0; ++q) slot(wave * P0 + q, 0, 2 * H0, 2 * H0, row1, m0, off0[q], dst0[q]);
  };
  auto point1 = [&] {
    int m0, n0, row1, rows;
    tile_of(w1.vb, m0, n0, row1, rows);
    w1.a = A + (size_t)m0 * lda;
#pragma unroll
    for (int q = 0; q < P1; ++q) slot(wave * P1 + q, H0 * 16, (row1 >> 3) - 2 * H0, ((rows - row1) >> 3) - 2 * H0, row1, m0, off1[q], dst1[q]);
  };
  const unsigned lds0 = lds_addr(dsmem);
  auto to = [&](unsigned stage, unsigned dst) { return lds0 + (S::SPARE && dst == S::SCRATCH ? dst : stage + dst); };
  auto advance = [&](Way& w, auto&& point) {
    if (++w.kt < nkt) return;
    if (w.vb + step < nblk) { w.vb += step; w.kt = kt0; point(); }
    else w.kt = nkt - 1;          // behind the last tile: copies that nobody reads
  };
  auto issue0 = [&](unsigned stage) {                 // stage: its byte offset
#pragma unroll
    for (int q = 0; q < P0; ++q) glds16_base(w0.a + (size_t)w0.kt * BK, off0[q], to(stage, dst0[q]));
#pragma unroll
    for (int q = 0; q < PB; ++q) glds16_base(W8 ? bbase[q] + (size_t)w0.kt * 512 : bbase[q >> 1] + (size_t)w0.kt * 1024 + (q & 1) * 512, lane * 16u, lds0 + stage + (S::A_UNITS + (wave * PB + q) * 64) * 16u);
    advance(w0, point0);
  };
  auto issue1 = [&](unsigned stage) {
#pragma unroll
    for (int q = 0; q < P1; ++q) glds16_base(w1.a + (size_t)w1.kt * BK, off1[q], to(stage, dst1[q]));
    advance(w1, point1);
  };
  point0();
  point1();
  if (kt0 < nkt) {
#pragma unroll
    for (int p = 0; p < NSTAGE; ++p) {
      issue0((unsigned)(p * STAGE) * 16u);
      if (p + 1 < NSTAGE) issue1((unsigned)(p * STAGE) * 16u);
    }
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
  __builtin_amdgcn_s_barrier();
  if (wm) __builtin_amdgcn_s_barrier();               // the second wave of a SIMD: one slot behind
  const int boff = S::A_UNITS + (wn * NT * (W8 ? 1 : 2)) * 64 + lane;
  int st = 0;                      // stage of the k-tile that is multiplied
  bool all_stored = false;         // the last epilogue issued NSTORE stores in this wave
  auto run = [&](auto mt_c, int m0, int n0, int my_row0) {      // one tile
    constexpr int MTW = decltype(mt_c)::value, MA = MTW > 0 ? MTW : 1, R0 = MTW > 0 ? H0 : 0, R1 = MTW - R0, RF = R0 > R1 ? R0 : R1;
    int aoff[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) aoff[kk] = ((wm ? S::ROW1 : 0) + li) * 8 + ((W8 ? g * 2 + kk : kk * 4 + g) ^ (li & 7));
    f32x4 acc[MA][NT];
#pragma unroll
    for (int i = 0; i < MA; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 fa[2][RF > 0 ? RF : 1], fb[2][NT];
    auto slot_end = [] {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    auto landed = [&](int kt) {     // what the next phase reads has landed and this one's fragments are in registers
      if (all_stored && kt - kt0 < NSTAGE - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LATER + S::NSTORE) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LATER) : "memory");
    };
    auto multiply = [&](auto from_c, auto n_c) {
      constexpr int from = decltype(from_c)::value, n = decltype(n_c)::value;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[from + i][j] = EPI == EPI_VIT_V ? mfma16(fa[kk][i], fb[kk][j], acc[from + i][j]) : mfma16(fb[kk][j], fa[kk][i], acc[from + i][j]);
    };
    for (int kt = kt0; kt < nkt; ++kt) {
      const u32x4* s = dsmem + st * STAGE;
      const unsigned cur = (unsigned)(st * STAGE) * 16u, before = (unsigned)((st == 0 ? NSTAGE - 1 : st - 1) * STAGE) * 16u;
      st = st == NSTAGE - 1 ? 0 : st + 1;
      if constexpr (MTW > 0) {
        if constexpr (W8) {
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const u32x4 raw = s[boff + j * 64];
            fb[0][j] = fp8x8_to_bf16x8(raw[0], raw[1]);
            fb[1][j] = fp8x8_to_bf16x8(raw[2], raw[3]);
          }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          if constexpr (!W8) {
#pragma unroll
            for (int j = 0; j < NT; ++j) fb[kk][j] = as_bf16x8(s[boff + (j * 2 + kk) * 64]);
          }
#pragma unroll
          for (int i = 0; i < R0; ++i) fa[kk][i] = as_bf16x8(s[aoff[kk] + i * 128]);
        }
      }
      issue1(before);
      landed(kt);
      slot_end();
      if constexpr (MTW > 0) multiply(std::integral_constant<int, 0>{}, std::integral_constant<int, R0>{});
      slot_end();
      if constexpr (MTW > 0) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int i = 0; i < R1; ++i) fa[kk][i] = as_bf16x8(s[aoff[kk] + (R0 + i) * 128]);
      }
      issue0(cur);
      landed(kt);
      slot_end();
      if constexpr (MTW > 0) multiply(std::integral_constant<int, R0>{}, std::integral_constant<int, R1>{});
      if (kt + 1 < nkt) slot_end();
    }
    if (kt0 < nkt && wm == 0) slot_end();
    unsigned char* const elds = reinterpret_cast<unsigned char*>(dsmem) + S::EPILOGUE + wave * (S::EGR * 2048);
    int l = lane;          // opaque: the epilogue's addresses are formed here and not kept in registers through the k-loop
    asm volatile("" : "+v"(l));
    if constexpr (VIT) {
      slot_end();                             // the slot in which the second wave of a SIMD multiplies for the last time
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();          // every wave is done with the stages, and its DMA pieces have landed
      if constexpr (EPI == EPI_VIT_V) {
        if constexpr (MTW > 0) vit_v_epilogue<MA, NT>(acc, m0 + my_row0, n0 + wn * 64, li, g, bias, M, N, vq);
      } else {
        // cos / sin rows of this tile: rows m0 .. m0 + BM - 1 of the [P, 40] fp32 tables are one contiguous piece of BM * 10 16-byte units each; reads
        // past the last row are clamped (those rows are never stored)
        constexpr int UNITS = BM * 10;
        const long first = (long)m0 * 10, last = (long)M * 10 - 1;
        for (int t = wave; t * 64 < UNITS; t += 8) {
          const long u = min(first + t * 64 + lane, last);
          glds16((vq.cs + u * 4), lds_addr(dsmem + t * 64));
          glds16((vq.sn + u * 4), lds_addr(dsmem + UNITS + t * 64));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        const float* lcs = reinterpret_cast<const float*>(dsmem);
        if constexpr (MTW > 0) vit_qk_epilogue<MA, NT>(acc, m0 + my_row0, n0 + wn * 64, my_row0, li, g, bias, C, ldc, M, N, vq.E, lcs, lcs + UNITS * 4);
      }
      return;
    } else if constexpr (MTW > 0 && EPI == EPI_PARTIAL) {
      tile_slab_wide<MTW, NT, 1, S::EGR * 2>(acc, m0 + my_row0, n0 + wn * 64, l, M, N, partial, W8 ? wscale : nullptr, elds);
    } else if constexpr (MTW > 0) {
      if (wide_rows<EPI>(C, ldc, bias, residual, ldr))
        tile_epilogue_wide<EPI, MTW, NT, S::EGR>(acc, m0 + my_row0, n0 + wn * 64, l, bias, residual, ldr, C, ldc, M, N, W8 ? wscale : nullptr, elds);
      else tile_epilogue<EPI, MTW, NT>(acc, m0 + my_row0, n0 + wn * 64, (n0 + wn * 64) / 2, l & 15, l >> 4, bias, residual, ldr, C, ldc, M, N, partial, W8 ? wscale : nullptr);
    }
    if (kt0 < nkt && wm == 1) slot_end();
  };
  for (int vb = vb0; vb < nblk; vb += step) {
    int m0, n0, row1, rows;
    tile_of(vb, m0, n0, row1, rows);
    const int my_row0 = wm ? row1 : 0;
    if (m0 + my_row0 >= M) run(std::integral_constant<int, 0>{}, m0, n0, my_row0);          // ragged last row tile: feed the ring only
    else if (S::VH && (wm ? rows - row1 : row1) == S::MTX * 16) run(std::integral_constant<int, S::MTX>{}, m0, n0, my_row0);
    else run(std::integral_constant<int, S::MT>{}, m0, n0, my_row0);
    all_stored = m0 + rows <= M && n0 + BN <= N;
  }
  if constexpr (VIT) return;
  if (!wm) __builtin_amdgcn_s_barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the copies behind the last tile: this block's LDS until they have landed
}
template <int BM, int EPI, bool W8>
__global__ __launch_bounds__(512) void gemm_walk_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias,
                                                        const bf16_t* __restrict__ residual, int ldr, bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m,
                                                        int tiles_n, float* __restrict__ partial, int kt_per_split, int raster, const float* __restrict__ wscale) {
  gemm_walk_body<BM, EPI, W8>(A, lda, W, bias, residual, ldr, C, ldc, M, N, K, tiles_m, tiles_n, partial, kt_per_split, raster, VitQkvEpi(), 0, 0, wscale);
}
// the vision tower's q|k|v projection (EPI_VIT_QK, EPI_VIT_V; EPI_VIT_QKV: both, N = 3E and 2E % 256 == 0): a tile a block
template <int BM, int EPI>
__global__ __launch_bounds__(512) void gemm_vit_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias,
                                                       bf16_t* __restrict__ C, int ldc, int M, int N, int K, int tiles_m, int tiles_n, VitQkvEpi vq, int raster) {
  const int nblk = tiles_m * tiles_n;
  for (int vb = blockIdx.x; vb < nblk; vb += gridDim.x) {     // one tile per block, or a persistent walk under the grid cap
    const int q = nblk >> 3, r = nblk & 7, xcd = vb & 7, bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (vb >> 3);
    int tn, tm;                                               // tile order: see gemm_big_kernel
    if (raster > 0) {
      const int band = bid / (raster * tiles_m), rem = bid - band * raster * tiles_m;
      const int bw = min(raster, tiles_n - band * raster);
      tm = rem / bw;
      tn = band * raster + (rem - tm * bw);
    } else {
      tn = bid / tiles_m;
      tm = bid - tn * tiles_m;
    }
    if constexpr (EPI == EPI_VIT_QKV) {
      // the column tiles of q and k run the rotation body, those of V the swapped-operand body on rows 2E.. of the packed weight
      const int qk_tiles = (2 * vq.E) >> 8;
      if (tn >= qk_tiles)
        gemm_walk_body<BM, EPI_VIT_V>(A, lda, W + (size_t)2 * vq.E * K, bias != nullptr ? bias + 2 * vq.E : nullptr, nullptr, 0, nullptr, 0, M, vq.E, K, 1, 1, nullptr, 0, 0,
                                      vq, tm, tn - qk_tiles);
      else
        gemm_walk_body<BM, EPI_VIT_QK>(A, lda, W, bias, nullptr, 0, C, ldc, M, 2 * vq.E, K, 1, 1, nullptr, 0, 0, vq, tm, tn);
    } else {
      gemm_walk_body<BM, EPI>(A, lda, W, bias, nullptr, 0, C, ldc, M, N, K, 1, 1, nullptr, 0, 0, vq, tm, tn);
    }
    if (vb + (int)gridDim.x < nblk) __syncthreads();          // the next tile's DMA reuses the stages (and the rotation's tables)
  }
}
template <int EPI>          // variable rows
__global__ __launch_bounds__(512) void gemm_walk_vh_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias,
                                                           const bf16_t* __restrict__ residual, int ldr, bf16_t* __restrict__ C, int ldc, int M, int N, int K,
                                                           int tiles_m, int tiles_n, float* __restrict__ partial, int kt_per_split, int raster) {
  gemm_walk_body<272, EPI>(A, lda, W, bias, residual, ldr, C, ldc, M, N, K, tiles_m, tiles_n, partial, kt_per_split, raster);
}

// ------------------------------------------------------------------------------------------------
// row tiles of 8 or 9 fragments (128 / 144 rows) for the split-K projections of ONE streaming chunk
// ------------------------------------------------------------------------------------------------
// M = 386 = 25 fragments: 3 row tiles of 9 + 8 + 8 instead of gemm_big_kernel<128>'s 4, whose fourth holds 2 rows.  A wave multiplies 4 or 5 row fragments x 4
// column fragments, 2 activation pieces per wave + an extra slot (rows 128-143, waves 0-1), a ring of THREE 51,200-B stages (one more tile in flight: at
// 32-40 MFMAs per wave and k-tile a single stage of look-ahead left the DMA round trip exposed: 104 vs 72 us).  One tile a block: its launches are one round.
// Accumulation order per output element = gemm_big_kernel's.  Requires packed bf16 W, K % 64 == 0, F >= 8, F <= 9 * floor(F / 8).
__global__ __launch_bounds__(512) void gemm_vh_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, int M, int N, int K, int tiles_m,
                                                      int tiles_n, float* __restrict__ partial, int kt_per_split, int raster) {
  constexpr int BN = 256, BK = 64, NT = 4;
  constexpr int MTX = 5, MTL = 4;                            // row fragments of an M-wave: MTL or MTX
  constexpr int APW = 2;                                     // 8-row activation pieces per wave below XBASE
  constexpr int XBASE = APW * 64;                            // the rows above ride on the extra slot
  constexpr int AROWS = XBASE + 16;
  constexpr int NSLOT = APW + 5;
  constexpr int A_UNITS = AROWS * 8;              // 16-byte units of the activation image
  constexpr int STAGE = A_UNITS + 32 * 64;        // + 32 W sub-tiles of 1 KB: 51,200 B
  constexpr int NST = 3;                          // ring depth: the k-step is too short to hide a DMA round trip behind one stage
  constexpr unsigned SCRATCH = (unsigned)NST * STAGE * 16u;  // byte offset of the 1-KB scratch behind the stages
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];

  const int nblk = tiles_m * tiles_n;
  for (int vb = blockIdx.x; vb < nblk; vb += gridDim.x) {     // one tile per block, or a persistent walk under the grid cap
  int bid = vb;
  {
    const int q = nblk >> 3, r = nblk & 7, xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  int tn, tm;                                     // tile order: see gemm_big_kernel
  if (raster > 0) {
    const int band = bid / (raster * tiles_m), rem = bid - band * raster * tiles_m;
    const int bw = min(raster, tiles_n - band * raster);
    tm = rem / bw;
    tn = band * raster + (rem - tm * bw);
  } else {
    tn = bid / tiles_m;
    tm = bid - tn * tiles_m;
  }
  const int F = (M + 15) >> 4, fbase = F / tiles_m, frem = F - fbase * tiles_m;
  const int f = fbase + (tm < frem ? 1 : 0);                       // row fragments of this tile: 8..9
  const int m0 = (tm * fbase + min(tm, frem)) << 4, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int li = lane & 15, g = lane >> 4;
  const int K32 = K >> 5, nfrag = N >> 4;
  const int f0 = f >> 1;                                           // M-wave 0: f0 fragments, M-wave 1: the rest
  const int my_mt = wm ? f - f0 : f0, my_row0 = wm ? f0 * 16 : 0;
  const bool wave_has_rows = m0 + my_row0 < M;

  // DMA piece table of this wave: slots 0-1 activation rows (wave*2 + q)*8 .. +7, slot 2 rows 128 + wave*8 .. (waves 0-1, if the tile
  // has them), slots 3-6 W sub-tiles wave*4 + q (n-fragment row st >> 1, 32-k block st & 1)
  const bf16_t* psrc[NSLOT];
  unsigned pdst[NSLOT];
  const int swz = ((lane & 7) ^ (lane >> 3)) << 3;
#pragma unroll
  for (int q = 0; q < APW; ++q) {
    const int row = (wave * APW + q) * 8 + (lane >> 3);
    psrc[q] = A + (size_t)min(m0 + row, M - 1) * lda + swz;
    pdst[q] = (unsigned)(wave * APW + q) * 1024u;
  }
  {
    const bool have = wave < 4 && XBASE + wave * 8 < f * 16;       // wave-uniform
    const int row = XBASE + (wave & 3) * 8 + (lane >> 3);
    psrc[APW] = have ? A + (size_t)min(m0 + row, M - 1) * lda + swz : A;
    pdst[APW] = have ? (unsigned)(XBASE / 8 + wave) * 1024u : SCRATCH;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int st = wave * 4 + q, fr = min((n0 >> 4) + (st >> 1), nfrag - 1);
    psrc[APW + 1 + q] = W + ((size_t)fr * K32 + (st & 1)) * 512 + lane * 8;
    pdst[APW + 1 + q] = (unsigned)(A_UNITS + st * 64) * 16u;
  }
  const unsigned lds0 = lds_addr(dsmem);
  auto piece = [&](int q, int kt, unsigned stage_lds) {             // q <= APW: activations advance 64 elements per k-tile, W 1024
    glds16(psrc[q] + (size_t)kt * (q <= APW ? BK : 1024), pdst[q] == SCRATCH ? lds0 + SCRATCH : stage_lds + pdst[q]);
  };

  const int nkt_all = K / BK;
  const int kt0 = blockIdx.y * kt_per_split, nkt = min(nkt_all, kt0 + kt_per_split);
  if (kt0 < nkt) {      // tiles kt0 .. kt0 + NST - 2 (clamped) into stages 0 .. NST - 2
#pragma unroll
    for (int p = 0; p < NST - 1; ++p)
#pragma unroll
      for (int q = 0; q < NSLOT; ++q) piece(q, min(kt0 + p, nkt - 1), lds0 + (unsigned)(p * STAGE) * 16u);
  }
  int aoff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) aoff[kk] = (my_row0 + li) * 8 + ((kk * 4 + g) ^ (li & 7));
  const int boff = A_UNITS + (wn * NT * 2) * 64 + lane;

  auto run = [&](auto mt_c) {
    constexpr int MTW = decltype(mt_c)::value;
    f32x4 acc[MTW > 0 ? MTW : 1][NT];
#pragma unroll
    for (int i = 0; i < (MTW > 0 ? MTW : 1); ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    int st_cur = 0;                   // stage of tile kt = (kt - kt0) % NST
    for (int kt = kt0; kt < nkt; ++kt) {
      // every wave issues exactly NSLOT pieces per tile, so the newest tile's pieces may stay in flight across the barrier
      static_assert(NSLOT == 7, "the counted wait below is written for 7 pieces per tile");
      asm volatile("s_waitcnt vmcnt(7)" ::: "memory");
      __builtin_amdgcn_s_barrier();   // tile kt complete in LDS; every wave is done reading tile kt-1
      const u32x4* s = dsmem + st_cur * STAGE;
      // the pieces of tile kt+NST-1 go out unconditionally (a branch would cut the scheduling region): past the last tile the source is
      // clamped and the copy lands in a stage nobody reads any more (the stage of tile kt-1)
      const int kt_dma = min(kt + NST - 1, nkt - 1);
      const int st_dma = st_cur == 0 ? NST - 1 : st_cur - 1;
      const unsigned dma_lds = lds0 + (unsigned)(st_dma * STAGE) * 16u;
      st_cur = st_cur == NST - 1 ? 0 : st_cur + 1;
      if constexpr (MTW == 0) {
#pragma unroll
        for (int q = 0; q < NSLOT; ++q) piece(q, kt_dma, dma_lds);
      } else {
        // pinned software pipeline of the fragment reads (gemm_big_kernel SCHED 6): the 8 W fragments of the k-tile up front, the
        // activation fragments through a 3-register ring two steps ahead, one DMA piece behind each of the first 9 row-tile steps
        bf16x8 fb[2][NT], fa[3];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int j = 0; j < NT; ++j) fb[kk][j] = as_bf16x8(s[boff + (j * 2 + kk) * 64]);
        fa[0] = as_bf16x8(s[aoff[0]]);
        fa[1] = as_bf16x8(s[aoff[0] + 128]);
#pragma unroll
        for (int t = 0; t < 2 * MTW; ++t) {
          if (t + 2 < 2 * MTW) fa[(t + 2) % 3] = as_bf16x8(s[aoff[(t + 2) / MTW] + ((t + 2) % MTW) * 128]);
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[t % MTW][j] = mfma16(fb[t / MTW][j], fa[t % 3], acc[t % MTW][j]);
          if (t < NSLOT) piece(t < NSLOT ? t : 0, kt_dma, dma_lds);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * NT + 2, 0);
#pragma unroll
        for (int t = 0; t < 2 * MTW; ++t) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the clamped copies of the last iteration
    __builtin_amdgcn_s_barrier();          // every wave is done with the stages, and its DMA pieces have landed
    if constexpr (MTW > 0)
      tile_slab_wide<MTW, NT>(acc, m0 + my_row0, n0 + wn * 64, lane, M, N, partial, nullptr, reinterpret_cast<unsigned char*>(dsmem) + wave * 8192);
  };
  using I0 = std::integral_constant<int, 0>;
  using IL = std::integral_constant<int, MTL>;
  using IX = std::integral_constant<int, MTX>;
  static_assert(2 * MTL >= NSLOT, "one DMA piece per row-tile step");
  if (!wave_has_rows) run(I0{});
  else if (my_mt == MTX) run(IX{});
  else run(IL{});
  if (vb + (int)gridDim.x < nblk) __syncthreads();     // the next tile's DMA reuses the stages
  }
}

// ------------------------------------------------------------------------------------------------
// tiled GEMM v4 ("tall"): ONE block row covers all of M (up to 448: a single-stream streaming chunk is 386 rows), 8 waves,
// (4 MT x 16) x 160 x 64 block tile, LDS-DMA for both operands, the two waves of a SIMD taking turns (gemm_walk_kernel)
// ------------------------------------------------------------------------------------------------
// Why: M = 386 on 128 x 256 tiles is 4 row tiles (the fourth holds 2 rows) x 148 = 592 blocks = 2.3 rounds of the 256 CUs.  Here every block owns ALL
// rows and 160 columns, so N = 37888 is 237 blocks = ONE round on 92.5 % of the CUs, and the W panel of a block is read once.
//   * waves: 4 (M) x 2 (N).  M-wave wm owns MT = ceil(fragments / 4) row fragments from wm * MT on; N-wave 0 owns column tiles 0-5, N-wave 1 tiles 6-9
//     (gate/up pairs stay inside a wave: SwiGLU epilogue).  Waves w and w + 4 share a SIMD: 6 + 4 column tiles of the same rows.
//   * a k-tile is two phases of row fragments (MT 7: three, 3 + 2 + 2 -- the weight fragments of a k-tile, 48 registers, stay for all of them); what a phase
//     reads is filled again behind it, in the order in which it is needed, as in gemm_walk_kernel.  (Phases for the two 32-k halves, 13 fragments each, with the
//     activations asked for one k-tile ahead: 103 us at 386 rows, but 108 / 103 at 448 and 73 / 67 at 192.)
//   * LDS: A image rows x 128 B (XOR-swizzled 16-byte chunks) + W tile 20 fragment sub-tiles of 1 KB = 77,824 B per stage (MT 7); two stages, with few rows up to four:
//     there the weights' way from HBM is what a launch takes.
// [37888, 3584] with SwiGLU, us, both waves in step (and always seven fragments) -> here: 100 rows 86 -> 57, 192 90 -> 67, 256 101 -> 74, 300 108 -> 84, 386 114 -> 106, 448 119 -> 107.
// Rows beyond M hold copies of the last ones: their products go into rows that are not stored.
// Requires packed W, K % 64 == 0.  W8: fp8 weights in their packed order, converted behind the LDS read, beside the other wave's MFMAs; their scale in the epilogue.
template <int MT, bool W8>
struct Tall {
  static constexpr int NP = MT > 6 ? 3 : 2, ROWS = 4 * MT * 16, A_UNITS = ROWS * 8;
  static constexpr int B_SUB = W8 ? 10 : 20, PB = (B_SUB + 7) / 8, STAGE = A_UNITS + B_SUB * 64;      // fragment sub-tiles of 1 KB (W8: a fragment's 64 k); 16-byte units
  static constexpr int frags(int p) { return NP == 3 ? (p == 0 ? 3 : 2) : (p == 0 ? (MT + 1) / 2 : MT / 2); }      // row fragments of phase p, = a wave's pieces of 8 rows
  static constexpr int from(int p) { return p == 0 ? 0 : p == 1 ? frags(0) : frags(0) + frags(1); }
  static constexpr int pieces(int p) { return frags(p) + (p == 0 ? PB : 0); }
  static constexpr int NSTAGE = 163840 / (STAGE * 16) > 4 ? 4 : 163840 / (STAGE * 16);
  // pieces that may be on their way when phase p ends: those of the NP NSTAGE - 2 parts asked for behind what the next phase reads
  static constexpr int later(int p) { int n = 0; for (int e = 0; e < NP * NSTAGE - 2; ++e) n += pieces((p + 2 + e) % NP); return n; }
  static constexpr size_t LDS = (size_t)NSTAGE * STAGE * 16;
  static_assert(NSTAGE >= 2 && (NP == 2 || MT == 7) && later(0) <= 63 && later(1) <= 63 && later(NP - 1) <= 63, "");
};
template <int EPI, int MT, bool W8>
__global__ __launch_bounds__(512) void gemm_tall_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
    const bf16_t* __restrict__ bias, const bf16_t* __restrict__ residual, int ldr,
    bf16_t* __restrict__ C, int ldc, int M, int N, int K, const float* __restrict__ wscale) {
  using T = Tall<MT, W8>;
  constexpr int BN = 160, BK = 64, NT0 = 6, NP = T::NP;
  extern __shared__ __attribute__((aligned(16))) u32x4 dsmem[];

  const int n0 = blockIdx.x * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;
  const int li = lane & 15, g = lane >> 4;
  const int K32 = K >> 5, nfrag = N >> 4, nkt = K / BK;
  const unsigned lds0 = lds_addr(dsmem), row_bytes = (unsigned)lda * 2u;

  // A wave's pieces of 8 rows: an offset per lane, the same for all of them but the one that ends at row M - 1, and a scalar one.  Pieces behind that one copy it
  // again, each to its own place: another phase's rows may still be read.
  const unsigned swz = ((lane & 7) ^ (lane >> 3)) << 4, whole = (unsigned)(lane >> 3) * row_bytes + swz;
  const int last = (M - 1) & ~7;
  const unsigned ends = (unsigned)min(lane >> 3, M - 1 - last) * row_bytes + swz;
  auto rows_part = [&](auto pc, int kt, int stage) {          // of phase p
    constexpr int p = decltype(pc)::value, n = T::frags(p);
    const bf16_t* base = A + (size_t)min(kt, nkt - 1) * BK;
#pragma unroll
    for (int q = 0; q < n; ++q) {
      const int x = wave * n + q, wr = x / (2 * n), to = wr * (MT * 16) + T::from(p) * 16 + (x - wr * 2 * n) * 8, row = min(to, last);
      glds16_base(base, (row == last ? ends : whole) + (unsigned)row * row_bytes, lds0 + (unsigned)(stage * T::STAGE) * 16u + to * 128u);
    }
  };
  auto weights = [&](int kt, int stage) {
    const int k = min(kt, nkt - 1);
#pragma unroll
    for (int q = 0; q < T::PB; ++q) {
      const int st = min(wave + 8 * q, T::B_SUB - 1);         // bf16: fragment row st >> 1, 32-k block st & 1
      const int fr = min((n0 >> 4) + (W8 ? st : st >> 1), nfrag - 1);
      const bf16_t* src = W8 ? W + (size_t)fr * (K >> 6) * 512 : W + ((size_t)fr * K32 + (st & 1)) * 512;
      glds16_base(src + (size_t)k * (W8 ? 512 : 1024), (unsigned)lane * 16u, lds0 + (unsigned)(stage * T::STAGE + T::A_UNITS + st * 64) * 16u);
    }
  };
  auto part = [&](auto pc, int kt, int stage) {
    if constexpr (decltype(pc)::value == 0) weights(kt, stage);
    rows_part(pc, kt, stage);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, NP - 1>;
#pragma unroll
  for (int k = 0; k < T::NSTAGE; ++k) {
    part(I0{}, k, k);
    if (NP == 3 || k + 1 < T::NSTAGE) part(I1{}, k, k);
    if constexpr (NP == 3) { if (k + 1 < T::NSTAGE) part(I2{}, k, k); }
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(T::later(NP - 1)) : "memory");
  __builtin_amdgcn_s_barrier();
  if (wn) __builtin_amdgcn_s_barrier();          // the second wave of a SIMD: one slot behind

  int aoff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) aoff[kk] = (wm * (MT * 16) + li) * 8 + ((W8 ? g * 2 + kk : kk * 4 + g) ^ (li & 7));
  const int boff = T::A_UNITS + (wn * NT0 * (W8 ? 1 : 2)) * 64 + lane;
  const int nbase = n0 + wn * NT0 * 16;
  auto run = [&](auto ntw_c) {
    constexpr int NTW = decltype(ntw_c)::value;
    f32x4 acc[MT][NTW];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NTW; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 fb[2][NTW], fa[2][T::frags(0)];
    auto slot_end = [] {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    auto read = [&](auto pc, const u32x4* s) {
      constexpr int p = decltype(pc)::value;
      if constexpr (p == 0) {
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
          if constexpr (W8) {
            const u32x4 raw = s[boff + j * 64];
            fb[0][j] = fp8x8_to_bf16x8(raw[0], raw[1]);
            fb[1][j] = fp8x8_to_bf16x8(raw[2], raw[3]);
          } else {
            fb[0][j] = as_bf16x8(s[boff + (j * 2) * 64]);
            fb[1][j] = as_bf16x8(s[boff + (j * 2 + 1) * 64]);
          }
        }
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < T::frags(p); ++i) fa[kk][i] = as_bf16x8(s[aoff[kk] + (T::from(p) + i) * 128]);
    };
    auto landed = [&](auto pc) {                 // what the next phase reads has landed and this one's fragments are in registers
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(T::later(decltype(pc)::value)) : "memory");
      slot_end();
    };
    auto multiply = [&](auto pc) {
      constexpr int p = decltype(pc)::value;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < T::frags(p); ++i)
#pragma unroll
          for (int j = 0; j < NTW; ++j) acc[T::from(p) + i][j] = mfma16(fb[kk][j], fa[kk][i], acc[T::from(p) + i][j]);
    };
    int st = 0;                                  // stage of the k-tile
    for (int kt = 0; kt < nkt; ++kt) {
      const int before = st == 0 ? T::NSTAGE - 1 : st - 1;
      const u32x4* s = dsmem + st * T::STAGE;
      read(I0{}, s);
      part(I2{}, kt + T::NSTAGE - 1, before);    // into what the last phase of the k-tile before has read
      landed(I0{});
      multiply(I0{});
      slot_end();
      read(I1{}, s);
      part(I0{}, kt + T::NSTAGE, st);
      landed(I1{});
      multiply(I1{});
      if constexpr (NP == 3) {
        slot_end();
        read(I2{}, s);
        part(I1{}, kt + T::NSTAGE, st);
        landed(I2{});
        multiply(I2{});
      }
      st = st == T::NSTAGE - 1 ? 0 : st + 1;
      if (wn == 0 || kt + 1 < nkt) slot_end();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the copies behind the last k-tile: this block's LDS until they have landed
    int le = lane;
    asm volatile("" : "+v"(le));          // the epilogue's addresses are formed here, not carried through the loop
    const int lie = le & 15, ge = le >> 4;
    if constexpr (W8) {                   // the rows' scales, one column tile at a time
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        asm volatile("" ::: "memory");
        const f32x4 sc = *reinterpret_cast<const f32x4*>(wscale + min(nbase + j * 16 + ge * 4, N - 4));
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][j] *= sc;
      }
    }
    tile_epilogue<EPI, MT, NTW>(acc, wm * (MT * 16), nbase, nbase / 2, lie, ge, bias, residual, ldr, C, ldc, M, N, nullptr, nullptr);
  };
  if (wn == 0) run(std::integral_constant<int, NT0>{});
  else run(std::integral_constant<int, 10 - NT0>{});
}

// 0: register-staged 2-stage kernel; 1: LDS-DMA 3-stage kernel; 2 (default): measured best per tile shape --
// 64-row tiles (72 KB ring, 2 blocks/CU) take the LDS-DMA kernel (1.5-1.6x), 128-row tiles keep the register-staged
// kernel (64 KB, 2 blocks/CU; the 96 KB ring would leave 1 block/CU and measured 0.75x).
static int g_gemm_variant = 2;
static int g_gemm_sched = 1;   // fragment-read schedule of gemm_big_kernel: 0 compiler order, 1 pinned software pipeline
void set_gemm_variant(int v);

static inline int raster_for(int tiles_m);
template <int EPI, bool W8>
static void launch_mid_w(const GemmArgs& a, hipStream_t st) {
  const int tiles_m = (a.M + 127) / 128, tiles_n = (a.N + 127) / 128, nkt = a.K / 64, S = (EPI == EPI_PARTIAL) ? a.nsplit : 1;
  constexpr size_t lds = (size_t)MID_STAGES * (16384 + (W8 ? 8192 : 16384));
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_mid_kernel<EPI, W8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  gemm_mid_kernel<EPI, W8><<<dim3(capped_grid((long)tiles_m * tiles_n), S), dim3(512), lds, st>>>(
      a.A, a.lda, a.W, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.partial, (nkt + S - 1) / S, a.wscale, raster_for(tiles_m), a.vq);
}
template <int EPI>
static void launch_mid(const GemmArgs& a, hipStream_t st) { a.w_fp8 ? launch_mid_w<EPI, true>(a, st) : launch_mid_w<EPI, false>(a, st); }
// The 64 x 128 tile.  Compute units left over by its blocks fetch weights ahead of them (strip_fetch): a block passes on some 50 B/ns and a step of the others takes
// 0.32 us, so that N / 60 blocks (fp8: N / 120) keep ahead of them from the first step on; fewer take the k-tiles at the end that they reach in time, under two
// fifths of them none (a run of its own, 1456 x 1280, K 5120, us: none 33.5, 16 blocks 32.2, 26 28.8; all of 390 x 3584, K 3584 on 16 blocks 42, on 60 20.5, none 22.4).
static int strip_fetch_blocks(int tiles, int N, int S, int nkt, bool w8, int* fetch) {
  const int idle = get_grid_cap() > 0 ? 0 : (256 - tiles * S) / S;
  const long reach = (long)idle * (w8 ? 120 : 60) * nkt / N;      // k-tiles of a split
  *fetch = (int)std::min<long>(reach, nkt);
  return idle > 0 && *fetch * 5 >= nkt * 2 ? idle : 0;
}
template <int EPI, bool W8>
static void launch_strip_w(const GemmArgs& a, hipStream_t st) {
  const int tiles_m = (a.M + 63) / 64, tiles_n = (a.N + 127) / 128, S = (EPI == EPI_PARTIAL) ? a.nsplit : 1, nkt = (a.K / 64 + S - 1) / S;
  const long tiles = (long)tiles_m * tiles_n;
  int fetch = 0;
  const int extra = tiles * S < 256 ? strip_fetch_blocks((int)tiles, a.N, S, nkt, W8, &fetch) : 0;
  constexpr size_t lds = (size_t)STRIP_STAGES * 8192;
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_strip_kernel<EPI, W8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  gemm_strip_kernel<EPI, W8><<<dim3(capped_grid(tiles) + extra, S), dim3(256), lds, st>>>(
      a.A, a.lda, a.W, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.partial, nkt, a.wscale, raster_for(tiles_m), fetch, a.vq);
}
template <int EPI>
static void launch_mid64(const GemmArgs& a, hipStream_t st) { a.w_fp8 ? launch_strip_w<EPI, true>(a, st) : launch_strip_w<EPI, false>(a, st); }
template <int BM, int EPI>
static void launch_tiled(const GemmArgs& a, hipStream_t st) {
  if constexpr (BM == 64) {
    if ((g_gemm_variant == 2 || g_gemm_variant == 7) && a.w_packed && (a.K & 63) == 0) return launch_mid64<EPI>(a, st);
  }
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + 127) / 128;
  const int nkt = (a.K + 63) / 64, S = (EPI == EPI_PARTIAL) ? a.nsplit : 1;
  if (g_gemm_variant == 1 || ((g_gemm_variant == 2 || g_gemm_variant == 7) && BM == 64)) {   // 7: auto without the 8-wave kernel
    constexpr size_t lds = (size_t)3 * ((BM / 16) * 2 + 16) * 1024;   // 96 KB (BM 128) / 72 KB (BM 64)
    static DeviceOnce attr_set;   // per instantiation
    if (attr_set.first()) {
      (void)hipFuncSetAttribute((const void*)gemm_glds_kernel<BM, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    }
    gemm_glds_kernel<BM, EPI><<<dim3(capped_grid((long)tiles_m * tiles_n), S), dim3(256), lds, st>>>(
        a.A, a.lda, a.W, a.ldw, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.w_packed, a.partial,
        (nkt + S - 1) / S);
    return;
  }
  gemm_tiled_kernel<BM, EPI><<<dim3(tiles_m * tiles_n, S), dim3(256), 0, st>>>(
      a.A, a.lda, a.W, a.ldw, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.w_packed, a.partial,
      (nkt + S - 1) / S);
}

// LCC_GEMM_RASTER (A/B, read once): band width of the tile order of the 8-wave kernels (bands of G column tiles walked row-major: the ~32
// tiles an XCD runs at a time form a (32 / G) x G super-tile), 0 = column-major (rounds 2-4)
static int g_gemm_raster = [] { const char* v = getenv("LCC_GEMM_RASTER"); return v ? atoi(v) : -1; }();
// -1 (default): bands of 4 column tiles once there are more than 6 row tiles; with few row tiles column-major already puts every row
// tile of a W panel side by side (M = 1131: 335 us column-major vs 342-355 us in bands, profiles/r05/gemm_vh_raster_ab.jsonl)
static inline int raster_for(int tiles_m) { return g_gemm_raster >= 0 ? g_gemm_raster : (tiles_m > 6 ? 4 : 0); }
template <int BM, int EPI, int SCHED, bool W8>
static void launch_big_s(const GemmArgs& a, hipStream_t st) {
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + 255) / 256;
  const int nkt = a.K / 64, S = (EPI == EPI_PARTIAL) ? a.nsplit : 1;
  // bf16: 128 KB (BM 256, 2 stages) / 144 KB (BM 128, 3 stages); fp8 W: 144 KB (BM 256) / 96 KB (BM 128), 3 stages
  constexpr size_t lds = (size_t)((BM >= 192 && !W8) ? 2 : 3) * (BM * 8 + (W8 ? 1024 : 2048)) * 16;
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) {
    (void)hipFuncSetAttribute((const void*)gemm_big_kernel<BM, EPI, SCHED, W8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  }
  gemm_big_kernel<BM, EPI, SCHED, W8><<<dim3(capped_grid((long)tiles_m * tiles_n), S), dim3(512), lds, st>>>(
      a.A, a.lda, a.W, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.partial, (nkt + S - 1) / S, a.wscale,
      raster_for(tiles_m));
}
// the walking kernels' offsets inside a tile are 32-bit (288 activation rows)
static bool walk_offsets_fit(const GemmArgs& a) { return (size_t)a.lda * 576 <= 0xffffffffu; }
// blocks of one split: one a tile while all splits' tiles fit the chip at once, else as many as it has units for
static unsigned walk_grid(long tiles, int S) { return tiles * S <= 256 ? capped_grid(tiles) : std::min(capped_grid(tiles), (unsigned)std::max(8, (256 / S) & ~7)); }
template <int BM, int EPI, bool W8>
static void launch_walk(const GemmArgs& a, hipStream_t st) {
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + 255) / 256;
  const int nkt = a.K / 64, S = (EPI == EPI_PARTIAL) ? a.nsplit : 1;
  constexpr size_t lds = Walk<BM, EPI, W8>::LDS;      // 256 / 192 / 160 / 128 rows: 160 / 145 / 137 / 160 KB; fp8 weights 128 / 113 / 105 / 112 KB
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_walk_kernel<BM, EPI, W8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  const unsigned grid = walk_grid((long)tiles_m * tiles_n, S);
  gemm_walk_kernel<BM, EPI, W8><<<dim3(grid, S), dim3(512), lds, st>>>(a.A, a.lda, a.W, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m,
                                                                       tiles_n, a.partial, (nkt + S - 1) / S, raster_for(tiles_m), a.wscale);
}
template <int BM, int EPI>
static void launch_vit_rows(const GemmArgs& a, hipStream_t st) {
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + 255) / 256;
  constexpr size_t lds = Walk<BM, EPI == EPI_VIT_QKV ? EPI_VIT_QK : EPI>::LDS;
  static_assert(BM * 320 <= Walk<BM, EPI_VIT_QK>::SCRATCH, "the rotation's tables in the stages");
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_vit_kernel<BM, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  gemm_vit_kernel<BM, EPI><<<dim3(capped_grid((long)tiles_m * tiles_n)), dim3(512), lds, st>>>(a.A, a.lda, a.W, a.bias, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.vq,
                                                                                              raster_for(tiles_m));
}
template <int EPI>
static void launch_vit(const GemmArgs& a, int rows, hipStream_t st) {
  if (rows == 256) launch_vit_rows<256, EPI>(a, st);
  else if (rows == 192) launch_vit_rows<192, EPI>(a, st);
  else launch_vit_rows<128, EPI>(a, st);
}
// variable-height row tiles: floor(F / 16) row tiles or fewer for F = ceil(M / 16) row fragments (small class: F / 8)
static bool vh_legal(const GemmArgs& a, bool small = false) {
  const int F = (a.M + 15) >> 4, t = F >> (small ? 3 : 4);
  return a.w_packed && !a.w_fp8 && (a.K % 64) == 0 && t >= 1 && F <= (small ? 9 : 18) * t && (a.N & 15) == 0 && walk_offsets_fit(a);
}
// Row tiles of an automatic choice: F / 18 to F / 16.  A tile of 17 / 18 fragments takes 1.08 / 1.17 of a 256-row tile's time (gate/up of 3,436 rows: 12 tiles of
// 17.9 fragments are 6.94 rounds, 642 us; 13 of 16.5 are 7.52, 663)
struct VhTiles { int tiles_m; float score; };
static VhTiles vh_tiles(int M, int N, int S) {
  const int F = (M + 15) >> 4;
  VhTiles best{F >> 4, 0.f};
  if (g_gemm_variant == 14) return best;
  for (int t = (F + 17) / 18; t <= F >> 4; ++t) {
    const int top = (F + t - 1) / t;
    const long blocks = (long)t * ((N + 255) / 256) * S;
    const float score = (top == 16 ? 1.f : top == 17 ? 0.985f : 0.96f) * (float)M / (float)(t * top * 16) * (float)blocks / (float)((blocks + 255) / 256 * 256);
    if (score > best.score) best = {t, score};
  }
  return best;
}
template <int EPI>
static void launch_vh(const GemmArgs& a, hipStream_t st) {
  const int nkt = a.K / 64, S = (EPI == EPI_PARTIAL) ? a.nsplit : 1;
  const int tiles_m = vh_tiles(a.M, a.N, S).tiles_m, tiles_n = (a.N + 255) / 256;
  constexpr size_t lds = Walk<272, EPI>::LDS;      // stages, scratch, epilogue: 156,672 B
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_walk_vh_kernel<EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  g_launch_counts[LC_GEMM_VH]++;
  const unsigned grid = walk_grid((long)tiles_m * tiles_n, S);
  gemm_walk_vh_kernel<EPI><<<dim3(grid, S), dim3(512), lds, st>>>(
      a.A, a.lda, a.W, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, tiles_m, tiles_n, a.partial, (nkt + S - 1) / S, raster_for(tiles_m));
}
static void launch_vh_small(const GemmArgs& a, hipStream_t st) {      // split-K slabs
  const int F = (a.M + 15) >> 4, tiles_m = F >> 3, tiles_n = (a.N + 255) / 256;
  const int nkt = a.K / 64, S = a.nsplit;
  constexpr size_t lds = (size_t)3 * (144 * 8 + 2048) * 16 + 1024;      // 3 x 51,200 B + the scratch
  static DeviceOnce attr_set;
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_vh_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  g_launch_counts[LC_GEMM_VH]++;
  gemm_vh_kernel<<<dim3(capped_grid((long)tiles_m * tiles_n), S), dim3(512), lds, st>>>(a.A, a.lda, a.W, a.M, a.N, a.K, tiles_m, tiles_n, a.partial, (nkt + S - 1) / S,
                                                                                        raster_for(tiles_m));
}
template <int BM, int EPI>
static void launch_big(const GemmArgs& a, hipStream_t st) {
  // pinned fragment-read pipeline with the LDS-DMA pieces spread between the row-tile steps (SCHED 6, default since round 3:
  // bit-identical to the burst-behind-the-barrier order SCHED 1 -- tools/gemm_checksum.py -- and 1.6-3.3 % faster on the prefill
  // GEMMs, +0.6 / +0.8 % tokens/s at 1 / 8 streams, profiles/r03/gemm_sched_spread_dma.txt); LCC_GEMM_SCHED=1 restores SCHED 1
  static const int spread = [] { const char* v = getenv("LCC_GEMM_SCHED"); return (v && atoi(v) == 1) ? 0 : 1; }();
  if (g_gemm_sched && spread) {
    // 128-row tiles that fill one round at most have nothing to walk, and the walk's longer prologue shows: 4,006 x 1536, K 768 17.6 us there, 19.1 walked;
    // vision fc1 of one chunk 27.7 / 28.6.  (192 and 256 rows gain from the scalar addresses: 4096 x 3584, K 3584 fp32 105.9 -> 102.5.)
    const long tiles = (long)((a.M + BM - 1) / BM) * ((a.N + 255) / 256) * (EPI == EPI_PARTIAL ? a.nsplit : 1);
    // fp8 weights on 128 rows: a burst instead of pieces spread over the steps (386 x 37888 149 us against 155)
    if (!walk_offsets_fit(a)) a.w_fp8 ? launch_big_s<(BM == 128 ? 128 : 256), EPI, 1, true>(a, st) : launch_big_s<(BM == 160 ? 192 : BM), EPI, 1, false>(a, st);
    else if (BM == 128 && tiles <= 256) a.w_fp8 ? launch_big_s<128, EPI, 1, true>(a, st) : launch_big_s<128, EPI, 6, false>(a, st);
    else a.w_fp8 ? launch_walk<BM, EPI, true>(a, st) : launch_walk<BM, EPI, false>(a, st);
  }
  else if (a.w_fp8) launch_big_s<(BM == 128 ? 128 : 256), EPI, 1, true>(a, st);
  else if (g_gemm_sched) launch_big_s<(BM == 160 ? 192 : BM), EPI, 1, false>(a, st);
  else launch_big_s<(BM == 160 ? 192 : BM), EPI, 0, false>(a, st);
}
// 13 / 17: the 192- / 160-row tile wherever eligible (bf16 weights); 14: variable-height row tiles (gemm_vh_kernel) wherever legal, else as 3;
// 16: 128 x 128 tiles (gemm_mid_kernel) wherever eligible
// 15: the small variable-height class (8 / 9 fragments) for split-K slabs wherever legal, else as 4
void set_gemm_variant(int v) {
  g_gemm_variant = v;
  g_gemm_sched = (v == 5 || v == 6) ? 0 : 1;
}
static bool big_eligible(const GemmArgs& a) { return a.w_packed && (a.K % 64) == 0 && a.M > 16; }
static_assert(GEMM_EPI_VIT_QK == (int)EPI_VIT_QK && GEMM_EPI_VIT_V == (int)EPI_VIT_V && GEMM_EPI_VIT_QKV == (int)EPI_VIT_QKV, "kernels.h / common.h disagree");
// M > 64: up to 64 rows the plain projection runs on the weight-streaming kernels (another fp32 summation order, and the better shape for so
// few rows) -- the fused form takes over where the plain one is an MFMA tile kernel, so both forms give the same bits
bool gemm_vit_qkv_eligible(int M, int E, int K) { return K > 0 && (K % 64) == 0 && M > 64 && (M & 3) == 0 && E > 0 && (E & 31) == 0; }

// 0 = not the 8-wave kernel, else its BM.  Variants 3 / 4 (5 / 6) force BM 256 / 128 wherever the kernel is eligible.
// Auto (2): estimated relative throughput = row utilisation x wave quantisation x measured tile efficiency.  The 8-wave
// kernels run one block per CU (256 slots), the 4-wave 64-row kernel two (512 slots).  Measured on MI355X (7B shapes):
// 256x256 tiles ~1.05-1.1 PF, 128x256 ~0.9 PF, 64x128 ~0.55 PF when the grid fills the chip; with few blocks (qkv at
// M = 386: 72 blocks of 128x256) the small tile wins.
// small variable-height class: on unless LCC_GEMM_VH_SMALL=0; shapes = one block-row class of a streaming chunk (fragment count not a
// multiple of 8, at most 448 rows) -- the engine asks gemm_tiled_num_splits with the same predicate, so split count and tile agree
static bool vh_small_on() { static const int on = [] { const char* v = getenv("LCC_GEMM_VH_SMALL"); return v ? atoi(v) : 1; }(); return on != 0; }
static bool vh_small_shape(int M, int K) {
  const int F = (M + 15) >> 4, t = F >> 3;
  return M > 64 && M <= 448 && (K % 64) == 0 && t >= 1 && F <= 9 * t && (F & 7) != 0;
}
static float tile_score(int M, int N, int S, int BM, int BN, int slots, float eff, bool ragged_skip) {
  const long tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN, blocks = tm * tn * S;
  const int half = BM / 2, mh = (M + half - 1) / half * half;   // the 8-wave kernel skips an all-padding half tile (~25 % cost)
  const float rows = ragged_skip ? (float)mh + 0.25f * (float)(tm * BM - mh) : (float)(tm * BM);
  const float util = (float)M / rows;
  const float quant = (float)blocks / (float)((blocks + slots - 1) / slots * slots);
  return util * quant * eff;
}
static bool tiles_192_on() { static const int on = [] { const char* v = getenv("LCC_GEMM_192"); return v ? atoi(v) : 1; }(); return on != 0; }      // A/B: 0 = 256 / 128 rows
static bool vh_on() { static const int on = [] { const char* v = getenv("LCC_GEMM_VH"); return v ? atoi(v) : 1; }(); return on != 0; }
// Score of the best tile of S splits, for the search of a split count alone (gemm_tiled_num_splits).  Which tile runs leaves a result's bits as they are; into how
// many fp32 sums a contraction is cut does not, so the count has weights of its own, which stay when the tiles' are measured anew.
static float split_score(const GemmArgs& a, int S) {
  const float on192 = tiles_192_on() ? 1.f : 0.f;
  float best = std::max(std::max(std::max(tile_score(a.M, a.N, S, 256, 256, 256, 1.0f, true), tile_score(a.M, a.N, S, 192, 256, 256, on192 * 0.93f, true)),
                                 std::max(tile_score(a.M, a.N, S, 160, 256, 256, on192 * 0.90f, false), tile_score(a.M, a.N, S, 128, 256, 256, 0.85f, true))),
                        std::max(tile_score(a.M, a.N, S, 128, 128, 256, 0.70f, false), tile_score(a.M, a.N, S, 64, 128, 256, 0.48f, false)));
  const int F = (a.M + 15) >> 4, t = F >> 4;
  if (vh_on() && vh_legal(a) && (F & 15) != 0) {
    const long blocks = (long)t * ((a.N + 255) / 256) * S;
    best = std::max(best, (float)a.M / (float)(t * ((F + t - 1) / t) * 16) * (float)blocks / (float)((blocks + 255) / 256 * 256));
  }
  return best;
}
// BM 192 (round 4, bf16 weights): a 256-row tile leaves the chip partly idle whenever (M / 256) x (N / 256) falls just short of a round --
// the o / down projections of 8 co-scheduled chunks are M = 3088 x N = 3584 = 13 x 14 = 182 blocks on 256 CUs (29 % idle); 17 x 14 = 238
// blocks of 192 rows fill 93 % of one round at 3/4 of the tile time.
// Variable-height tiles (returned as 272): F / 18 to floor(F / 16) row tiles of 16-18 fragments (vh_tiles) -- scored with every tile as tall as the
// tallest, no ragged tile.
// Efficiencies against 256 rows: a round of [37888, 3584] takes 52 / 58 / 67 / 77.5 us with 128 / 160 / 192 / 256 rows and 82-85 / 91 with 17 / 18 fragments: 0.75, 0.84,
// 0.87, 1, 0.985, 0.96 (short tiles move more bytes from the L2 per product, and from 0.85 of the chip on power is the limit).  192 rows at 0.93 and 160 at 0.90 had
// been measured on tiles whose waves kept in step, us there / here: 3580 x 37888 722 / 701, 5000 x 3584, K 18944 590 / 464, 3994 x 17920, K 1536 181 / 169, 11648 x 1536,
// K 8960 278 / 225, 3994 x 4608 113 / 96, 1600 x 37888 372 / 341, 4096 x 14336 326 / 309; the worst of 28 shapes whose tile changed 1950 / 1973.
// (fp32 output, one slab: 4096 x 25088 672 / 603, 4096 x 14336 372 / 342, 5992 x 14336 531 / 477, 7920 x 7168 363 / 331.)
// LCC_GEMM_VH=0: rounds 2-4 tile choice.
// wide_only: 256-column tiles as they stand against a 64 x 128 one that dequantises fp8 weights first (gemm_w8)
static int big_tile_rows(const GemmArgs& a, int S, bool wide_only = false) {
  if (!big_eligible(a)) return 0;
  if (g_gemm_variant == 14) return vh_legal(a) ? 272 : 256;
  if (g_gemm_variant == 3 || g_gemm_variant == 5) return 256;
  if (g_gemm_variant == 4 || g_gemm_variant == 6) return 128;
  if (g_gemm_variant == 13) return wide_only ? 256 : 192;
  if (g_gemm_variant == 17) return wide_only ? 256 : 160;
  if (g_gemm_variant == 15) return (a.partial != nullptr && vh_small_shape(a.M, a.K) && vh_legal(a, true)) ? 144 : 128;
  if (g_gemm_variant == 16) return wide_only ? 128 : 129;
  if (g_gemm_variant != 2) return 0;
  const bool slabs = a.partial != nullptr && S > 1;
  const float s256 = tile_score(a.M, a.N, S, 256, 256, 256, 1.0f, true);
  const bool short_tiles = tiles_192_on() && !(a.w_fp8 && (slabs || wide_only));
  const float s192 = !short_tiles ? 0.f : tile_score(a.M, a.N, S, 192, 256, 256, 0.88f, true);
  // BM 160 (bf16 weights): where 192 rows start a last round that is mostly empty.  The vision proj / fc2 of 15,840 rows are 83 x 5 tiles of 192 rows =
  // 1.62 rounds; 99 x 5 of 160 fill 1.93 at 5/6 of the time each: proj 55.7 -> 52.1 us, fc2 201 -> 178.
  const float s160 = !short_tiles ? 0.f : tile_score(a.M, a.N, S, 160, 256, 256, 0.86f, false);
  // 128 rows: 0.85 us a step while all tiles run at once, 0.93 in several rounds (514 rows of [37888, 3584]: 192-row tiles 141 us, these 156; fp8 weights 136 / 160)
  const bool second_round = (long)((a.M + 127) / 128) * ((a.N + 255) / 256) * S > 256;
  const float s128 = tile_score(a.M, a.N, S, 128, 256, 256, second_round && !slabs && !wide_only ? 0.76f : a.w_fp8 ? 0.85f : 0.82f, true);
  // gemm_strip_kernel / gemm_mid_kernel: 0.38 (0.33 since its waves read their own weights) / 0.52 us a step of 64 x 128 / 128 x 128 against 0.85 of 128 x 256, one tile a compute
  // unit at a time.  With 0.33 the choice is within 4 % of the best in 223 of 230 shapes, 5 to 7 % off in the others: the weights stay (two 64-row
  // tiles side by side take twice as long).  Returned as 0 / 129.  The 128-row form wins where its blocks fill one round and the 64-row
  // form's need two; beyond a round the 256-column tiles do (shapes around the lines: 1000 x 3584, K 3584: 43 / 34 / 52 us for 64 x 128 /
  // 128 x 128 / 128 x 256; 1456 x 3584: 73 / 61 / 52; 520 x 3584: 25 / 33 / 50).  With fp8 weights the steps stand alike (4608, K 3584: 386 rows
  // 25 / 33 / 49, 600 rows 42 / 34 / 50, 1000 rows 73 / 61 / 49; 200 x 3584, K 18944 in four splits 68 / 48 / 66).
  const float s64 = wide_only ? tile_score(a.M, a.N, S, 64, 128, 512, 0.55f, false) : tile_score(a.M, a.N, S, 64, 128, 256, 0.48f, false);
  const float s128m = wide_only ? 0.f : tile_score(a.M, a.N, S, 128, 128, 256, 0.70f, false);
  if (vh_on() && vh_legal(a) && (((a.M + 15) >> 4) & 15) != 0) {      // F % 16 == 0: the 256-row tiles are the same thing
    const float svh = vh_tiles(a.M, a.N, S).score;
    if (svh > s256 && svh > s192 && svh > s160 && svh > s128 && svh > s128m && svh > s64) return 272;
  }
  // small class (returned as 144): split-K slabs of one streaming chunk's projections, where the 128-row tiles leave a nearly empty last row tile
  if (vh_small_on() && a.partial != nullptr && vh_small_shape(a.M, a.K) && vh_legal(a, true)) {
    const int F = (a.M + 15) >> 4, t = F >> 3, maxf = (F + t - 1) / t;
    const long blocks = (long)t * ((a.N + 255) / 256) * S;
    const float svs = 0.85f * (float)a.M / (float)(t * maxf * 16) * (float)blocks / (float)((blocks + 255) / 256 * 256);
    if (svs > s256 && svs > s192 && svs > s160 && svs > s128 && svs > s128m && svs > s64) return 144;
  }
  if (s256 >= s192 && s256 >= s160 && s256 >= s128 && s256 >= s128m && s256 >= s64) return 256;
  if (s192 >= s160 && s192 >= s128 && s192 >= s128m && s192 >= s64) return 192;
  if (s160 > s128 && s160 > s128m && s160 > s64) return 160;
  // a last row tile that is half empty saves nothing while all blocks run at once beside full ones, and two 64-row tiles a unit hide each other's ends:
  // at 129 to 192 rows [17920, 1536] 19.1 us against 23.0 with 128 x 256 tiles, [4608, 3584] in four splits 15.4 / 16.6, [3584, 3584] in six 13.3 / 14.2.
  // Up to 24 steps a block: [3584, 18944] in six splits (49 steps) 51.7 / 44.4
  const bool one_round = a.M > 128 && (long)((a.M + 127) / 128) * ((a.N + 255) / 256) * S <= 256 && a.K <= 64 * 24 * S;
  const float s128_64 = one_round && !a.w_fp8 ? tile_score(a.M, a.N, S, 128, 256, 256, 0.85f, false) : s128;
  if (s128 >= s128m && s128_64 >= s64) return 128;
  return s128m > s64 ? 129 : 0;
}

// The tall kernel serves one-block-row problems whose column tiles fill most of ONE round of the chip (7B gate/up at a streaming
// chunk: 237 blocks).  Variant 8 forces it wherever it is legal (tests).
// (fp8 weights with a residual would need more registers than a wave has; a row's offset, up to 448 rows from A, is 32-bit)
static bool tall_legal(const GemmArgs& a) {
  return big_eligible(a) && !(a.w_fp8 && a.epilogue == EPI_RESIDUAL) && a.M <= 448 && (a.N & 15) == 0 && (size_t)a.lda * 896 <= 0xffffffffu;
}
static bool tall_wanted(const GemmArgs& a) {
  if (!tall_legal(a)) return false;
  if (g_gemm_variant == 8) return true;
  if (g_gemm_variant != 2) return false;
  const int blocks = (a.N + 159) / 160;
  if (blocks < 192 || blocks > 256) return false;
  // without SwiGLU: [37888, 3584] with bias, us, other tiles / these: 256 rows 82 / 102, 288 100 / 86, 340 110 / 95, 448 123 / 108; fp8 weights, which have one height there (launch_tall_w):
  // 256 72 / 102, 300 98 / 104, 386 113 / 107
  if (a.epilogue != EPI_SWIGLU) return a.M > (a.w_fp8 ? 384 : 256);
  // Up to 256 rows where the other tiles (128 x 128, or two rows of 128 x 256) are more than one round.  K 3584 with SwiGLU, us, other tiles / these:
  //   bf16, N 37888: 65 rows 67 / 55, 128 71 / 59, 192 80 / 67, 256 89 / 74, 272 and more 84 / 84 (walking tiles; 300 rows 101 before them);  N 30720: 100 rows 48 / 52, 256 67 / 67
  //   fp8,  N 37888: 65 to 128 rows 56 / 57, 129 105 / 68, 256 90 / 75, 272 110 / 87, 330 114 / 96;  N 30720: 100 rows 44 / 56, 256 61 / 73
  return a.M > 256 || (a.N > 32768 && a.M > (a.w_fp8 ? 128 : 64));
}
template <int EPI, int MT, bool W8>
static void launch_tall_rows(const GemmArgs& a, hipStream_t st) {
  constexpr size_t lds = Tall<MT, W8>::LDS;
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) (void)hipFuncSetAttribute((const void*)gemm_tall_kernel<EPI, MT, W8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  gemm_tall_kernel<EPI, MT, W8><<<dim3((a.N + 159) / 160), dim3(512), lds, st>>>(a.A, a.lda, a.W, a.bias, a.residual, a.ldr, a.C, a.ldc, a.M, a.N, a.K, a.wscale);
}
template <int EPI, bool W8>
static void launch_tall_w(const GemmArgs& a, hipStream_t st) {
  // fragments for each quarter of the rows, where such rows come here unforced (tall_wanted); [37888, 3584] with bias, us, always seven / these: 272 rows 102 / 86, 300 103 / 87, 340 105 / 95
  constexpr bool few = EPI == EPI_SWIGLU;
  const int mt = ((a.M + 15) / 16 + 3) / 4;
  if constexpr (few) {
    if (mt <= 2) return launch_tall_rows<EPI, 2, W8>(a, st);
    if (mt == 3) return launch_tall_rows<EPI, 3, W8>(a, st);
    if (mt == 4) return launch_tall_rows<EPI, 4, W8>(a, st);
  }
  if constexpr (few || !W8) {
    if (mt == 5) return launch_tall_rows<EPI, 5, W8>(a, st);
    if (mt == 6) return launch_tall_rows<EPI, 6, W8>(a, st);
  }
  launch_tall_rows<EPI, 7, W8>(a, st);
}
template <int EPI>
static void launch_tall(const GemmArgs& a, hipStream_t st) {
  g_launch_counts[LC_GEMM_TALL]++;
  if constexpr (EPI != EPI_RESIDUAL) {
    if (a.w_fp8) return launch_tall_w<EPI, true>(a, st);
  }
  launch_tall_w<EPI, false>(a, st);
}

template <int EPI>
static void launch_tiled_bm(const GemmArgs& a, hipStream_t st) {
  if constexpr (EPI != EPI_PARTIAL) {       // split-K slabs stay on the 128/256-row tiles (the tall kernel has no K split)
    if (tall_wanted(a)) return launch_tall<EPI>(a, st);
  }
  const int big = big_tile_rows(a, 1);
  if (big == 129) return launch_mid<EPI>(a, st);
  if (big == 272) return launch_vh<EPI>(a, st);
  if (big == 256) return launch_big<256, EPI>(a, st);
  if (big == 192) return launch_big<192, EPI>(a, st);
  if (big == 160) return launch_big<160, EPI>(a, st);
  if (big == 128) return launch_big<128, EPI>(a, st);
  // 128-row tiles only for large M with a grid that fills the chip; otherwise 64-row tiles (less waste on a ragged M such as
  // 386 rows, more blocks, and the faster LDS-DMA kernel)
  const long blocks128 = (long)((a.M + 127) / 128) * ((a.N + 127) / 128);
  if (a.M >= 1024 && blocks128 >= 512) launch_tiled<128, EPI>(a, st);
  else launch_tiled<64, EPI>(a, st);
}

// Which kernel family serves a packed-weight GEMM of this shape under the current variant (host logic only: no launch, no GPU needed):
// 16 = weight-streaming GEMV, 448 = tall, 272 / 144 = variable-height tiles (big / small class), 256 / 192 / 160 / 128 = the 8-wave tile of
// that height x 256 columns, 129 = 128 x 128, 64 = 64 x 128.  `nsplit` > 0: the split-K slab form with that many splits (as the engine asks: gemm_tiled_num_splits).
int gemm_plan(int M, int N, int K, int epilogue, int nsplit, bool w_fp8) {
  GemmArgs a; a.M = M; a.N = N; a.K = K; a.w_packed = 1; a.w_fp8 = w_fp8 ? 1 : 0; a.epilogue = epilogue; a.nsplit = nsplit;
  static float dummy;
  if (nsplit > 0) a.partial = &dummy;      // never dereferenced here: only "is this the slab form?"
  const bool skinny = gemm_routes_skinny(M, K, w_fp8) && epilogue != EPI_QUICK_GELU && epilogue != EPI_GELU_ERF && epilogue != EPI_RESIDUAL;
  if (skinny) return 16;
  if (nsplit <= 0 && tall_wanted(a)) return 448;
  const int big = big_tile_rows(a, nsplit > 0 ? nsplit : 1);
  return big != 0 ? big : 64;
}

// ------------------------------------------------------------------------------------------------
// skinny GEMV-like kernel (M <= 64; MG = 1..4 activation fragments per weight fragment, two from ten rows on where a block takes several tiles): HBM-bound weight streaming
// ------------------------------------------------------------------------------------------------
// Block = 4 waves.  The block owns NTILE*16 consecutive W rows and the 64-element K chunks [c_begin, c_end) of split
// blockIdx.y; wave w takes chunks c_begin + w, + 4, ...  W fragments go HBM -> VGPR -> MFMA (no LDS: each byte is used
// once); per chunk and tile a lane issues two 16-byte loads plus the matching x fragment (L2/L1 resident).  The four
// partial accumulators are reduced through LDS and wave 0 runs the epilogue.  D'[n][m]: lane (m = l&15, g) ends with 4
// consecutive n for activation row m.
//
// W layouts:  row-major [N,K] (a wave load = 16 rows x 64 B), or PACKED [N/16][K/32][4 g][16 rows][8 k]: the 1-KB
// A-operand fragment of (row tile, 32-k block) is contiguous in lane order, so every wave load is one contiguous KB and a
// block streams one contiguous 16*K*2-byte region per tile -- linear DRAM streams instead of 64-byte row segments.
//
// PIPE 0: UNR chunks are loaded, then multiplied (latency hidden by ~20 resident waves per CU);
// PIPE 1: two-stage software pipeline (the next stage's loads are in flight while this one is multiplied).
__device__ unsigned int lcc_zero_page_g[64];  // 256 zero bytes: x operand of absent K chunks (address select, no branch)

// MG = 16-row groups of activations (M <= 16 * MG): the weight fragment of a k-block is loaded ONCE and multiplied with MG activation
// fragments (rows mg*16 + li), so 17..64 decode streams still read every weight byte once per step (round 4: before, they went through the
// 64-row GEMM tiles: 8.5-11.9 ms per 32-stream step where the weight stream alone costs ~2.6 ms).
// bx, split, nsplit: the block's weight tiles and its share of K.  red: the waves' sums; xs_all: the activations of MG > 1
template <int NTILE, int MODE, bool PACKED, int UNR, int PIPE, int MG>
LCC_DEVICE void gemv_skinny_body(
    const bf16_t* __restrict__ X, int ldx, const bf16_t* __restrict__ W, int ldw,
    const bf16_t* __restrict__ bias, void* __restrict__ out, int ldo, int M, int N, int K, int chunks_per_split, const GemvTail& tail, int bx, int split, int nsplit,
    f32x4 (*red)[NTILE * MG][64], u32x4* xs_all) {
  constexpr int NW = 4;
  static_assert(MODE != 3 || MG == 1, "the fused tail serves M <= 2");
  // MG > 1: the activation rows of a 64-k chunk are fetched in FULL 128-byte lines (one load instruction = 8 rows x 128 B; the
  // fragment-shaped load -- 16 rows x 64 B per instruction -- was 2.3x slower at M = 32: 99 vs 43 us for the gate/up GEMV,
  // profiles/r04/bench_32streams_mg_gemv_first_version.json) and turned into MFMA fragments through a wave-private LDS scratch with the
  // (chunk ^ row & 7) swizzle of gemm_big_kernel's activation image: ds_write_b128 of the raw lines, ds_read_b128 of the fragments.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  const int n0 = bx * (NTILE * 16);
  const int nchunk = (K + 63) >> 6, K32 = (K + 31) >> 5;
  const int cb = split * chunks_per_split, ce = min(nchunk, cb + chunks_per_split);

  // MG == 1: xp[0] = this lane's fragment slice (row li, 8 k of lane group g).  MG > 1: xp[i], i < 2 MG = line piece of instruction i:
  // row i*8 + (lane >> 3), 16-byte piece lane & 7 of the row's 128-byte chunk line (slots [h][mg] of the stage arrays hold i = h*MG + mg)
  const bf16_t* xp[MG > 1 ? 2 * MG : 1];
  if (MG == 1) {
    xp[0] = X + (size_t)min(li, M - 1) * ldx + g * 8;
  } else {
#pragma unroll
    for (int i = 0; i < 2 * MG; ++i) xp[i] = X + (size_t)min(i * 8 + (lane >> 3), M - 1) * ldx + (lane & 7) * 8;
  }
  const bf16_t* zp = reinterpret_cast<const bf16_t*>(lcc_zero_page_g) + (MG == 1 ? g * 8 : (lane & 7) * 8);
  u32x4* xs = xs_all + (MG > 1 ? wave * MG * 128 : 0);
  const bf16_t* wp[NTILE];
#pragma unroll
  for (int t = 0; t < NTILE; ++t)
    wp[t] = PACKED ? W + (size_t)min((n0 >> 4) + t, ((N + 15) >> 4) - 1) * K32 * 512 + lane * 8      // a last block's absent tiles: the last one again, not stored
                   : W + (size_t)min(n0 + t * 16 + li, N - 1) * ldw + g * 8;

  f32x4 acc[NTILE][MG];
#pragma unroll
  for (int t = 0; t < NTILE; ++t)
#pragma unroll
    for (int mg = 0; mg < MG; ++mg) acc[t][mg] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // loads are unconditional (32-k block index clamped into range) so that the compiler emits straight-line loads with
  // counted waits; an absent block is cancelled by pointing the (shared) x fragment at a zero page.
  auto load_stage = [&](int c0, u32x4 (&wv)[UNR][2][NTILE], u32x4 (&xv)[UNR][2][MG]) {
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int cc = c0 + u * NW;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kb = 2 * cc + h;                        // 32-k block
        const bool ok = cc < ce && kb < K32;              // wave-uniform
        const int kbc = min(kb, K32 - 1);
#pragma unroll
        for (int t = 0; t < NTILE; ++t)
          wv[u][h][t] = __builtin_nontemporal_load((const u32x4*)(wp[t] + (size_t)kbc * (PACKED ? 512 : 32)));
        if (MG == 1) {
          xv[u][h][0] = ld16(ok ? xp[0] + kbc * 32 : zp);
        } else {       // full lines of the 64-k chunk (both k-blocks): instruction i = h*MG + mg; a chunk whose second k-block is past K reads the
                       // zero page for the whole chunk only when the chunk itself is absent (K % 64 == 32 never occurs with MG > 1: gemm_routes_skinny
                       // from 17 rows on, gemv_rows_tiles and gemv_rows_pair_ok below)
#pragma unroll
          for (int mg = 0; mg < MG; ++mg) xv[u][h][mg] = ld16((cc < ce) ? xp[h * MG + mg] + min(cc, nchunk - 1) * 64 : zp);
        }
      }
    }
  };
  auto mma_stage = [&](const u32x4 (&wv)[UNR][2][NTILE], const u32x4 (&xv)[UNR][2][MG]) {
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      u32x4 xf[2][MG];
      if (MG == 1) {
        xf[0][0] = xv[u][0][0];
        xf[1][0] = xv[u][1][0];
      } else {
        // raw lines -> wave-private LDS image [row][8 x 16 B], chunk c of row r at r*8 + (c ^ (r & 7)) -> fragments (row mg*16 + li,
        // k-block h, lane group g)
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < 2 * MG; ++i) {
          const int row = i * 8 + (lane >> 3);
          xs[row * 8 + ((lane & 7) ^ (row & 7))] = xv[u][i / MG][i % MG];
        }
        wave_lds_order();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int mg = 0; mg < MG; ++mg) xf[h][mg] = xs[(mg * 16 + li) * 8 + ((h * 4 + g) ^ (li & 7))];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NTILE; ++t)
#pragma unroll
          for (int mg = 0; mg < MG; ++mg) acc[t][mg] = mfma16(as_bf16x8(wv[u][h][t]), as_bf16x8(xf[h][mg]), acc[t][mg]);
    }
  };
  constexpr int STEP = UNR * NW;  // chunk stride of one stage
  if (PIPE == 0) {
    for (int c = cb + wave; c < ce; c += STEP) {
      u32x4 wa[UNR][2][NTILE], xa[UNR][2][MG];
      load_stage(c, wa, xa);
      mma_stage(wa, xa);
    }
  } else {
    u32x4 wa[UNR][2][NTILE], xa[UNR][2][MG], wb[UNR][2][NTILE], xb[UNR][2][MG];
    int c = cb + wave;
    load_stage(c, wa, xa);
    for (; c < ce; c += 2 * STEP) {
      // MG > 1: the issue order is PINNED (all loads of the next stage, then the whole current stage).  Left to itself hipcc sinks the next
      // stage's activation loads behind this stage's MFMAs and waits for them a few instructions later (vmcnt retires in order: the weight
      // loads issued before them are waited for too) -- the two-stage pipeline collapsed and the M = 32 gate/up GEMV ran at 2.8 TB/s
      // (98.8 us, profiles/r04/bench_32streams_mg_gemv_*.json)
      load_stage(c + STEP, wb, xb);
      if (MG > 1) __builtin_amdgcn_sched_barrier(0);
      mma_stage(wa, xa);
      if (MG > 1) __builtin_amdgcn_sched_barrier(0);
      load_stage(c + 2 * STEP, wa, xa);
      if (MG > 1) __builtin_amdgcn_sched_barrier(0);
      mma_stage(wb, xb);
      if (MG > 1) __builtin_amdgcn_sched_barrier(0);
    }
  }

  // cross-wave reduction
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < NTILE; ++t)
#pragma unroll
      for (int mg = 0; mg < MG; ++mg) red[wave - 1][t * MG + mg][lane] = acc[t][mg];
  }
  __syncthreads();
  if (MODE == 3) {
    // split-K slabs + FUSED TAIL.  Publish/consume protocol (cdna_hip_programming.md G16 R1, counter form): write-through (sc1)
    // slab stores -> vmcnt(0) -> __syncthreads -> one lane: relaxed agent fetch_add (ticket).  The block that draws the last
    // ticket: one lane agent-scope acquire -> __syncthreads -> plain loads of every slab.  Placement-independent.
    if (wave == 0) {
#pragma unroll
      for (int t = 0; t < NTILE; ++t)
#pragma unroll
        for (int w = 0; w < NW - 1; ++w) acc[t][0] += red[w][t * MG][lane];
      if (li < M) {
        float* o = (float*)out + ((size_t)split * M + li) * ldo;
#pragma unroll
        for (int t = 0; t < NTILE; ++t) {
          const int n = n0 + t * 16 + g * 4;
          if (n < N) {
            // write-through (sc1) slab stores: relaxed agent-scope 8-byte atomic stores lower to `global_store_dwordx2 sc0 sc1`,
            // so NO per-block release fence (buffer_wbl2) is needed -- measured: a release fence in each of the ~900 blocks
            // made the whole kernel ~17 us slower
            unsigned long long* p8 = reinterpret_cast<unsigned long long*>(o + n);
            const unsigned long long lo = (unsigned long long)__float_as_uint(acc[t][0][0]) | ((unsigned long long)__float_as_uint(acc[t][0][1]) << 32);
            const unsigned long long hi = (unsigned long long)__float_as_uint(acc[t][0][2]) | ((unsigned long long)__float_as_uint(acc[t][0][3]) << 32);
            __hip_atomic_store(p8, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(p8 + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every storing wave drains its write-through stores
    }
    __syncthreads();
    float* flag = reinterpret_cast<float*>(&red[0][0][0]);   // all LDS in ONE array
    if (threadIdx.x == 0) {
      const int ticket = __hip_atomic_fetch_add(tail.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      flag[0] = (ticket == (int)(gridDim.x * gridDim.y) - 1) ? 1.f : 0.f;
    }
    __syncthreads();
    if (flag[0] == 0.f) return;
    if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();
    if (tail.kind == 1) {
      for (int m = 0; m < M; ++m)
        tail_add_rmsnorm_row(tail.h + (size_t)m * N, (const float*)out, nsplit, (size_t)M * ldo, (size_t)m * ldo, tail.norm_w,
                             tail.y + (size_t)m * N, N, tail.eps, flag + 8);
    } else {
      RopeTailArgs ra{tail.bias, tail.cs, tail.sn, tail.tok_stream, tail.tok_pos, tail.kv_len, tail.kv_base, tail.lay, tail.layer,
                      tail.q_out, tail.n_q_heads};
      tail_rope_kv_append((const float*)out, nsplit, M, ra);
    }
    if (threadIdx.x == 0) __hip_atomic_store(tail.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
    return;
  }
  if (wave > 0) return;
#pragma unroll
  for (int t = 0; t < NTILE; ++t)
#pragma unroll
    for (int mg = 0; mg < MG; ++mg)
#pragma unroll
      for (int w = 0; w < NW - 1; ++w) acc[t][mg] += red[w][t * MG + mg][lane];

#pragma unroll
  for (int mg = 0; mg < MG; ++mg) {
    const int m = mg * 16 + li;
    if (m >= M) continue;
    if (MODE == 0) {
      float* o = (float*)out + ((size_t)split * M + m) * ldo;
#pragma unroll
      for (int t = 0; t < NTILE; ++t) {
        const int n = n0 + t * 16 + g * 4;
        if (n < N) *reinterpret_cast<f32x4*>(o + n) = acc[t][mg];
      }
    } else if (MODE == 1) {
      bf16_t* o = (bf16_t*)out + (size_t)m * ldo;
#pragma unroll
      for (int t = 0; t < NTILE; ++t) {
        const int n = n0 + t * 16 + g * 4;
        if (n >= N) continue;
        float v[4] = {acc[t][mg][0], acc[t][mg][1], acc[t][mg][2], acc[t][mg][3]};
        if (bias != nullptr) {
          u32x2 b = ld8(bias + n);
          v[0] += lo2f(b.x); v[1] += hi2f(b.x); v[2] += lo2f(b.y); v[3] += hi2f(b.y);
        }
        st8(o + n, (u32x2){pack2(v[0], v[1]), pack2(v[2], v[3])});
      }
    } else {  // swiglu: even tiles = 16 gate rows, the next one = the 16 matching up rows
      static_assert(MODE != 2 || NTILE % 2 == 0, "swiglu needs the gate and up tile in one block");
      bf16_t* o = (bf16_t*)out + (size_t)m * ldo;
#pragma unroll
      for (int t = 0; t + 1 < NTILE; t += 2) {
        if (n0 + t * 16 >= N) continue;
        float r[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = silu_bf16(rbf(acc[t][mg][q])) * rbf(acc[t + 1][mg][q]);
        st8(o + n0 / 2 + t * 8 + g * 4, (u32x2){pack2(r[0], r[1]), pack2(r[2], r[3])});
      }
    }
  }
}
constexpr int gemv_sums(int ntile, int mg) { return 3 * ntile * mg * 64; }      // 16-byte pieces of LDS
constexpr int gemv_rows_lds(int mg) { return mg > 1 ? 4 * mg * 128 : 1; }
template <int NTILE, int MODE, bool PACKED, int UNR, int PIPE, int MG = 1>
__global__ __launch_bounds__(256) void gemv_skinny_kernel(
    const bf16_t* __restrict__ X, int ldx, const bf16_t* __restrict__ W, int ldw,
    const bf16_t* __restrict__ bias, void* __restrict__ out, int ldo, int M, int N, int K, int chunks_per_split, GemvTail tail) {
  __shared__ f32x4 red[3][NTILE * MG][64];
  __shared__ u32x4 xs_all[gemv_rows_lds(MG)];
  gemv_skinny_body<NTILE, MODE, PACKED, UNR, PIPE, MG>(X, ldx, W, ldw, bias, out, ldo, M, N, K, chunks_per_split, tail, blockIdx.x, blockIdx.y, gridDim.y, red, xs_all);
}
// Two products of the same 9..64 rows in ONE launch: a gate/up projection (SwiGLU, NTILE tiles a block) and, behind its blocks, another one into fp32 slabs (a tile
// a block).  Alone, neither fills the chip (32 rows of the 2B layer-list decoder: 187 blocks of gate/up, 13.6 us; 162 of the input projection, 4.6 us): the
// small one runs on the units that the large one leaves, and a launch of the step is gone.  Same sums, same bits.
struct GemvPart { const bf16_t *X, *W; void* out; int ldx, ldo, N, K, cps; };
template <int NTILE, int MG>
__global__ __launch_bounds__(256) void gemv_rows_pair_kernel(GemvPart sw, GemvPart in, int M, int nb_sw, int nb_in) {
  constexpr int S1 = gemv_sums(NTILE, MG), S2 = gemv_sums(1, MG);
  __shared__ f32x4 red[S1 > S2 ? S1 : S2];
  __shared__ u32x4 xs_all[gemv_rows_lds(MG)];
  const int b = blockIdx.x;
  const GemvTail none{};
  if (b < nb_sw)
    gemv_skinny_body<NTILE, 2, true, 1, 1, MG>(sw.X, sw.ldx, sw.W, sw.K, nullptr, sw.out, sw.ldo, M, sw.N, sw.K, sw.cps, none, b, 0, 1,
                                               reinterpret_cast<f32x4(*)[NTILE * MG][64]>(red), xs_all);
  else
    gemv_skinny_body<1, 0, true, 1, 1, MG>(in.X, in.ldx, in.W, in.K, nullptr, in.out, in.ldo, M, in.N, in.K, in.cps, none, (b - nb_sw) % nb_in, (b - nb_sw) / nb_in, 1,
                                           reinterpret_cast<f32x4(*)[MG][64]>(red), xs_all);
}

static int g_skinny_rows = 64;
// THE predicate of the weight-streaming route (the engine used to decide it from its own copy of the row limit, so a forced tile
// variant or a K that is not a multiple of 64 could leave it handing GEMV-derived split counts to the tiled kernels): M rows against a
// [N, K] weight go through gemv_skinny_kernel / gemv_w8_kernel iff this holds (and the epilogue is one the GEMV kernels have).
bool gemm_routes_skinny(int M, int K, bool w_fp8) {
  if (w_fp8) return M <= 16;
  return M <= (g_gemm_variant == 2 ? g_skinny_rows : 16) && (K % 32 == 0) && (M <= 16 || K % 64 == 0);
}
int set_skinny_rows(int rows) { const int old = g_skinny_rows; g_skinny_rows = rows < 16 ? 16 : (rows > 64 ? 64 : rows); return old; }
static int g_gemv_variant = 1;  // 0: UNR2 single stage; 1: UNR1 two-stage pipeline (default: best measured); 2: UNR2 two-stage
void set_gemv_variant(int v) { g_gemv_variant = v; }

template <int NTILE, int MODE, bool PACKED, int MG>
static void launch_gemv_mg(dim3 grid, const GemmArgs& a, void* out, int ldo, int cps, hipStream_t st) {
  if constexpr (MG > 1) {     // 10..64 rows (the pair kernel: 9..64): the two-stage pipeline with one chunk per stage (register budget: NTILE x MG accumulators + MG x fragments)
    gemv_skinny_kernel<NTILE, MODE, PACKED, 1, 1, MG><<<grid, dim3(256), 0, st>>>(a.A, a.lda, a.W, a.ldw, a.bias, out, ldo, a.M, a.N, a.K, cps, a.tail);
    return;
  } else switch (g_gemv_variant) {
    case 1:
      gemv_skinny_kernel<NTILE, MODE, PACKED, 1, 1><<<grid, dim3(256), 0, st>>>(a.A, a.lda, a.W, a.ldw, a.bias, out, ldo, a.M, a.N, a.K, cps, a.tail);
      break;
    case 2:
      gemv_skinny_kernel<NTILE, MODE, PACKED, 2, 1><<<grid, dim3(256), 0, st>>>(a.A, a.lda, a.W, a.ldw, a.bias, out, ldo, a.M, a.N, a.K, cps, a.tail);
      break;
    default:
      gemv_skinny_kernel<NTILE, MODE, PACKED, 2, 0><<<grid, dim3(256), 0, st>>>(a.A, a.lda, a.W, a.ldw, a.bias, out, ldo, a.M, a.N, a.K, cps, a.tail);
  }
}
template <int NTILE, int MODE, bool PACKED>
static void launch_gemv(dim3 grid, const GemmArgs& a, void* out, int ldo, int cps, hipStream_t st) {
  const int mg = (a.M + 15) / 16;
  if (mg <= 1) launch_gemv_mg<NTILE, MODE, PACKED, 1>(grid, a, out, ldo, cps, st);
  else if (mg == 2) launch_gemv_mg<NTILE, MODE, PACKED, 2>(grid, a, out, ldo, cps, st);
  else if (mg == 3) launch_gemv_mg<NTILE, MODE, PACKED, 3>(grid, a, out, ldo, cps, st);
  else launch_gemv_mg<NTILE, MODE, PACKED, 4>(grid, a, out, ldo, cps, st);
}
template <int NTILE, int MODE>
static void launch_gemv_l(dim3 grid, const GemmArgs& a, void* out, int ldo, int cps, hipStream_t st) {
  if (a.w_packed) launch_gemv<NTILE, MODE, true>(grid, a, out, ldo, cps, st);
  else launch_gemv<NTILE, MODE, false>(grid, a, out, ldo, cps, st);
}

// 10..64 rows: a block of one 16-row weight tile reads more activations than weights (32 rows: twice as many bytes, and a compute unit pulls about 40
// GB/s of either), so packed weights go up to six tiles to a block.  What a unit then pulls: rounds of blocks x (tiles + 16-row groups of
// activations); more tiles only where that is clearly less, since their registers leave one or two waves a SIMD.  32 rows, [151936, 1536]: 116.5 us with
// one tile, 80.8 with four (5.8 TB/s); [152064, 3584] 261 -> 182; 64 rows: 358 -> 239.  Three tiles against one, two, four at 32 rows (a row of launches
// on weights from memory): [1536, 10496] in eight splits 9.7 / 11.7, 11.7, 10.3; [1536, 8960] in eight 9.0 / 12.0, 10.5, 9.6.  Six: [3584, 18944] in five
// 30.3 against 35.6 with two and 37.4 with four, [4608, 3584] in four 10.7 / 12.4 with one, gate/up with SwiGLU [17920, 1536] 14.1 / 16.2 with two,
// 64 rows of [37888, 3584] 68.6 / 76.0.  Where one tile's blocks fill a round at most it stays: [2048, 1536] in two splits 4.7 / 5.1.
// 10 to 16 rows run as 17 do, two groups of rows (one, in fragment-shaped loads: 2 to 6 % slower a step), whose way through LDS and larger last sums have to be earned: what a unit pulls,
// by the 64 k of a chunk, has to be less by 20 + 6 for each tile.  us, one tile / several (which), 10, 12, 14, 16 rows: [3584, 18944] in five (6) 26.8 / 25.3, 28.2 / 25.5, 29.4 / 25.6, 31.4 / 25.8;
// [152064, 3584] (4) 178 / 165, 190 / 166, 204 / 167, 219 / 168; [4608, 3584] in four (6) 8.9 / 9.5, 9.2 / 9.5, 9.5 / 9.5, 9.9 / 9.5; [4096, 4096] in four (2, 2, 4, 4) 7.9 / 8.6, 8.2 / 8.6, 8.5 / 9.1,
// 8.9 / 9.1; [2304, 1536] in two (2) 4.4 / 5.1, 4.6 / 5.1, 4.7 / 5.1, 4.9 / 5.1; of 216 such products (54 shapes) 56 were slower without this, by 2 to 18 %, five are with it, by 2 to 5.  With SwiGLU a
// block has two tiles anyway and two groups of rows come with four: no such line ([17920, 1536] (6) 13.4 / 12.8, 13.9 / 12.7, 14.1 / 12.9, 14.0 / 12.4, [12288, 2048] (4) 16 rows 11.8 / 10.9)
static int gemv_rows_tiles(const GemmArgs& a, int S) {
  const bool pairs = a.epilogue == EPI_SWIGLU;
  const int least = pairs ? 2 : 1;
  if (!a.w_packed || a.M <= 9 || (a.M <= 16 && (a.K & 63) != 0)) return least;
  const int tiles = (a.N + 15) / 16;
  auto cost = [&](int nt) { return (float)(((long)((tiles + nt - 1) / nt) * S + 255) / 256) * ((float)nt + (float)a.M / 16.f); };
  int nt = least;
  for (int c : {2, 3, 4, 6})
    if (c > least && !(pairs && (c & 1)) && cost(c) < (c == 2 ? 0.97f : 0.85f) * cost(nt)) nt = c;
  const int chunks = ((a.K + 63) / 64 + S - 1) / S;
  if (a.M <= 16 && !pairs && nt > least && (cost(least) - cost(nt)) * (float)chunks < 20.f + 6.f * (float)nt) return least;
  return nt;
}
// the weight tiles a block takes (0: another route), for packed weights; nsplit > 0: slabs
int gemv_plan_tiles(int M, int N, int K, int epilogue, int nsplit) {
  if (gemm_plan(M, N, K, epilogue, nsplit, false) != 16) return 0;
  GemmArgs a; a.w_packed = 1; a.M = M; a.N = N; a.K = K; a.epilogue = epilogue;
  return gemv_rows_tiles(a, std::max(nsplit, 1));
}
template <int NTILE, int MODE>
static void launch_gemv_tiles(const GemmArgs& a, int S, void* out, int ldo, int cps, hipStream_t st) {
  const dim3 grid((a.N + NTILE * 16 - 1) / (NTILE * 16), S);
  if (a.M <= 32) launch_gemv_mg<NTILE, MODE, true, 2>(grid, a, out, ldo, cps, st);
  else if (a.M <= 48) launch_gemv_mg<NTILE, MODE, true, 3>(grid, a, out, ldo, cps, st);
  else launch_gemv_mg<NTILE, MODE, true, 4>(grid, a, out, ldo, cps, st);
}
template <int MODE>
static void launch_gemv_rows(const GemmArgs& a, int S, void* out, int ldo, int cps, hipStream_t st) {
  constexpr int LEAST = MODE == 2 ? 2 : 1;
  switch (gemv_rows_tiles(a, S)) {
    case 6: launch_gemv_tiles<6, MODE>(a, S, out, ldo, cps, st); break;
    case 4: launch_gemv_tiles<4, MODE>(a, S, out, ldo, cps, st); break;
    case 3: if constexpr (MODE != 2) launch_gemv_tiles<3, MODE>(a, S, out, ldo, cps, st); break;
    case 2: if constexpr (MODE != 2) { launch_gemv_tiles<2, MODE>(a, S, out, ldo, cps, st); break; } [[fallthrough]];
    default: launch_gemv_l<LEAST, MODE>(dim3((a.N + 16 * LEAST - 1) / (16 * LEAST), S), a, out, ldo, cps, st);
  }
}

// (9 to 16 rows run as 17 here: the kernel has two groups of rows at least)
static int pair_tiles(const GemmArgs& sw) { GemmArgs a = sw; a.M = std::max(sw.M, 17); return gemv_rows_tiles(a, 1); }
// Whether one launch is the faster one.  Beside a small body (two tiles a block) it was in all shapes measured.  A large one leaves a unit to one block at a time,
// the input projection's blocks of one tile among them: what the units pull (gemv_rows_tiles), apart with the tiles each would take alone and together, and a
// launch's worth of it, 160, between them.  us a layer of a decode step, apart / together, width, feed-forward, query rank, rows:  1536, 8960, 768: 17 rows 59.8 / 56.4,
// 64 79.1 / 75.1;  3584, 18944, 1536: 17 124.6 / 122.4, 32 136.7 / 131.3, 64 168.9 / 162.8;  8192, 28672, 1536: 64 400 / 392;  3584, 8192, 3584: 48 128.3 / 128.3,
// 64 142.1 / 146.9;  8192, 14336, 4096: 32 191.3 / 189.4, 64 234.5 / 237.4;  8192, 8192, 4096: 17 134.9 / 134.7, 32 140.7 / 141.8, 64 172.1 / 181.0
static bool gemv_rows_pair_pays(const GemmArgs& in, const GemmArgs& sw) {
  const int nt = pair_tiles(sw), alone = gemv_rows_tiles(in, in.nsplit);
  if (nt == 2) return true;
  const float groups = (float)sw.M / 16.f;
  const long blocks_sw = (sw.N / 16 + nt - 1) / nt, blocks_in = (long)(in.N / 16) * in.nsplit, blocks_alone = (long)((in.N / 16 + alone - 1) / alone) * in.nsplit;
  const float chunks_in = (float)(((in.K + 63) / 64 + in.nsplit - 1) / in.nsplit);
  const float block_sw = ((float)nt + groups) * (float)((sw.K + 63) / 64), block_in = (1.f + groups) * chunks_in;
  const float sw_alone = (float)((blocks_sw + 255) / 256) * block_sw;
  const float apart = sw_alone + (float)((blocks_alone + 255) / 256) * ((float)alone + groups) * chunks_in;
  const float together = std::max(sw_alone, ((float)blocks_sw * block_sw + (float)blocks_in * block_in) / 256.f + block_in);
  return together - apart < 160.f;
}
// in: fp32 slabs (partial, nsplit); sw: SwiGLU.  Takes what the two calls of gemm_bf16 would take on the weight-streaming path with 9 to 64 rows, where it pays
bool gemv_rows_pair_ok(const GemmArgs& in, const GemmArgs& sw) {
  auto one = [](const GemmArgs& a) {
    return a.w_packed && !a.w_fp8 && a.M > 8 && a.M <= 64 && a.N > 0 && gemm_routes_skinny(a.M, a.K, false) && (a.K & 63) == 0 && (a.N & 15) == 0 && (a.lda & 7) == 0 &&
           (((uintptr_t)a.A | (uintptr_t)a.W) & 15) == 0 && a.bias == nullptr && a.tail.kind == 0;
  };
  return one(in) && one(sw) && in.M == sw.M && in.partial != nullptr && in.nsplit >= 1 && in.nsplit <= 8 && in.nsplit <= (in.K + 63) / 64 && in.epilogue == EPI_NONE &&
         sw.partial == nullptr && sw.epilogue == EPI_SWIGLU && (sw.N & 31) == 0 && (sw.ldc & 3) == 0 && ((uintptr_t)sw.C & 15) == 0 && gemv_rows_pair_pays(in, sw);
}
template <int NTILE>
static void launch_rows_pair(const GemmArgs& in, const GemmArgs& sw, hipStream_t st) {
  const int nin = (in.K + 63) / 64, nb_sw = (sw.N + NTILE * 16 - 1) / (NTILE * 16), nb_in = in.N / 16;
  const GemvPart a{sw.A, sw.W, sw.C, sw.lda, sw.ldc, sw.N, sw.K, (sw.K + 63) / 64}, b{in.A, in.W, in.partial, in.lda, in.N, in.N, in.K, (nin + in.nsplit - 1) / in.nsplit};
  const dim3 grid(nb_sw + nb_in * in.nsplit);
  if (in.M <= 32) gemv_rows_pair_kernel<NTILE, 2><<<grid, dim3(256), 0, st>>>(a, b, in.M, nb_sw, nb_in);
  else if (in.M <= 48) gemv_rows_pair_kernel<NTILE, 3><<<grid, dim3(256), 0, st>>>(a, b, in.M, nb_sw, nb_in);
  else gemv_rows_pair_kernel<NTILE, 4><<<grid, dim3(256), 0, st>>>(a, b, in.M, nb_sw, nb_in);
}
int gemv_rows_pair(const GemmArgs& in, const GemmArgs& sw, hipStream_t st) {
  if (!gemv_rows_pair_ok(in, sw)) return LCC_ERR_ARG;
  g_launch_counts[LC_GEMV_ROWS_PAIR]++;
  switch (pair_tiles(sw)) {
    case 6: launch_rows_pair<6>(in, sw, st); break;
    case 4: launch_rows_pair<4>(in, sw, st); break;
    default: launch_rows_pair<2>(in, sw, st);
  }
  return 0;
}

// ------------------------------------------------------------------------------------------------
// fp8 weights (OCP e4m3, per-output-row fp32 scale): decode GEMV, and the routes of every product
// ------------------------------------------------------------------------------------------------
// PACKED8 layout [N/16][K/64][4 g][16 rows][16 k] bytes: lane (g, row) of a 16-row x 64-k fragment owns the 16 consecutive
// k = kb*64 + g*16 .. +15 of its row, i.e. ONE 16-byte load per lane per fragment and 1 KB contiguous per wave load -- the same
// linear HBM stream as the bf16 packed layout at half the bytes.  The 16 bytes feed TWO 16x16x32 MFMAs (bytes 0-7, 8-15): the
// k -> MFMA-slot assignment is arbitrary as long as the activation fragment uses the same one (x[kb*64 + g*16 + 0..7] and
// + 8..15).  e4m3 -> bf16 is exact (v_cvt_pk_f32_fp8 + v_cvt_pk_bf16_f32), products accumulate in fp32, and the row scale is
// applied once to the fp32 sum -- so the result is the bf16 GEMV of the exactly dequantised integers times the scale.

template <int NTILE, int MODE>   // MODE 0 fp32 split-K slabs, 1 bf16 + bias, 2 SwiGLU (tile 0 = 16 gate rows, tile 1 = their up rows)
__global__ __launch_bounds__(256) void gemv_w8_kernel(
    const bf16_t* __restrict__ X, int ldx, const uint8_t* __restrict__ W, const float* __restrict__ wscale,
    const bf16_t* __restrict__ bias, void* __restrict__ out, int ldo, int M, int N, int K, int chunks_per_split) {
  constexpr int NW = 4, UNR = 2;
  __shared__ f32x4 red[NW - 1][NTILE][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (NTILE * 16);
  const int split = blockIdx.y;
  const int nchunk = K >> 6;
  const int cb = split * chunks_per_split, ce = min(nchunk, cb + chunks_per_split);
  const int nfrag = N >> 4;

  const bf16_t* xp = X + (size_t)min(li, M - 1) * ldx + g * 16;
  const bf16_t* zp = reinterpret_cast<const bf16_t*>(lcc_zero_page_g) + g * 16;
  const uint8_t* wp[NTILE];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) wp[t] = W + (size_t)min((n0 >> 4) + t, nfrag - 1) * nchunk * 1024 + lane * 16;

  f32x4 acc[NTILE];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  auto load_stage = [&](int c0, u32x4 (&wv)[UNR][NTILE], u32x4 (&xv)[UNR][2]) {
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int cc = c0 + u * NW;
      const bool ok = cc < ce;                          // wave-uniform
      const int ccl = min(cc, nchunk - 1);
#pragma unroll
      for (int t = 0; t < NTILE; ++t) wv[u][t] = __builtin_nontemporal_load((const u32x4*)(wp[t] + (size_t)ccl * 1024));
      const bf16_t* xs = ok ? xp + ccl * 64 : zp;       // an absent chunk is cancelled by a zero activation fragment
      xv[u][0] = ld16(xs);
      xv[u][1] = ld16(xs + 8);
    }
  };
  auto mma_stage = [&](const u32x4 (&wv)[UNR][NTILE], const u32x4 (&xv)[UNR][2]) {
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int t = 0; t < NTILE; ++t) {
        acc[t] = mfma16(fp8x8_to_bf16x8(wv[u][t][0], wv[u][t][1]), as_bf16x8(xv[u][0]), acc[t]);
        acc[t] = mfma16(fp8x8_to_bf16x8(wv[u][t][2], wv[u][t][3]), as_bf16x8(xv[u][1]), acc[t]);
      }
  };
  constexpr int STEP = UNR * NW;
  {
    u32x4 wa[UNR][NTILE], xa[UNR][2], wb[UNR][NTILE], xb[UNR][2];
    int c = cb + wave;
    load_stage(c, wa, xa);
    for (; c < ce; c += 2 * STEP) {
      load_stage(c + STEP, wb, xb);
      mma_stage(wa, xa);
      load_stage(c + 2 * STEP, wa, xa);
      mma_stage(wb, xb);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < NTILE; ++t) red[wave - 1][t][lane] = acc[t];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int t = 0; t < NTILE; ++t) {
#pragma unroll
    for (int w = 0; w < NW - 1; ++w) acc[t] += red[w][t][lane];
    acc[t] *= *reinterpret_cast<const f32x4*>(wscale + min(n0 + t * 16 + g * 4, N - 4));
  }
  if (li >= M) return;
  if (MODE == 0) {
    float* o = (float*)out + ((size_t)split * M + li) * ldo;
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      const int n = n0 + t * 16 + g * 4;
      if (n < N) *reinterpret_cast<f32x4*>(o + n) = acc[t];
    }
  } else if (MODE == 1) {
    bf16_t* o = (bf16_t*)out + (size_t)li * ldo;
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      const int n = n0 + t * 16 + g * 4;
      if (n >= N) continue;
      float v[4] = {acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
      if (bias != nullptr) {
        u32x2 b = ld8(bias + n);
        v[0] += lo2f(b.x); v[1] += hi2f(b.x); v[2] += lo2f(b.y); v[3] += hi2f(b.y);
      }
      st8(o + n, (u32x2){pack2(v[0], v[1]), pack2(v[2], v[3])});
    }
  } else {
    static_assert(MODE != 2 || NTILE == 2, "swiglu needs the gate and up tile in one block");
    bf16_t* o = (bf16_t*)out + (size_t)li * ldo;
    const int oc = n0 / 2 + g * 4;
    if (n0 < N) {
      float r[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] = silu_bf16(rbf(acc[0][q])) * rbf(acc[NTILE - 1][q]);
      st8(o + oc, (u32x2){pack2(r[0], r[1]), pack2(r[2], r[3])});
    }
  }
}

// layout probe (tests/test_gpu_ops.py::test_mfma_layout_probe): D[16x16] = A[16x32] * B[32x16] with the fragment maps of
// common.h, one wave.  Verifies the operand/result lane maps every kernel in this library relies on.
__global__ __launch_bounds__(64) void mfma_probe_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                        float* __restrict__ D) {
  const int l = threadIdx.x, i = l & 15, g = l >> 4;
  bf16_t av[8], bv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    av[e] = A[i * 32 + g * 8 + e];        // A[i][k = g*8+e]
    bv[e] = B[(g * 8 + e) * 16 + i];      // B[k = g*8+e][j = i]
  }
  u32x4 a = (u32x4){(unsigned)av[0] | ((unsigned)av[1] << 16), (unsigned)av[2] | ((unsigned)av[3] << 16),
                    (unsigned)av[4] | ((unsigned)av[5] << 16), (unsigned)av[6] | ((unsigned)av[7] << 16)};
  u32x4 b = (u32x4){(unsigned)bv[0] | ((unsigned)bv[1] << 16), (unsigned)bv[2] | ((unsigned)bv[3] << 16),
                    (unsigned)bv[4] | ((unsigned)bv[5] << 16), (unsigned)bv[6] | ((unsigned)bv[7] << 16)};
  f32x4 c = mfma16(as_bf16x8(a), as_bf16x8(b), (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int r = 0; r < 4; ++r) D[(g * 4 + r) * 16 + i] = c[r];  // D[row = g*4+r][col = i]
}
int mfma_probe(const bf16_t* A, const bf16_t* B, float* D, hipStream_t st) {
  mfma_probe_kernel<<<dim3(1), dim3(64), 0, st>>>(A, B, D);
  return 0;
}

// number of inter-block K splits of a skinny GEMV: enough blocks (x4 waves) to keep >= ~16 waves per CU in flight,
// every wave keeps >= ~3 64-element chunks, and the fp32 slab traffic stays small (S <= 8)
int gemv_num_splits(int N, int K) {
  // tuning knobs (debug): LCC_GEMV_TARGET = blocks aimed at (default 1024), LCC_GEMV_MINCHUNK = 64-k chunks per split at least (12)
  static const int target = [] { const char* e = getenv("LCC_GEMV_TARGET"); return e ? std::max(64, atoi(e)) : 1024; }();
  static const int minchunk = [] { const char* e = getenv("LCC_GEMV_MINCHUNK"); return e ? std::max(1, atoi(e)) : 12; }();
  const int tiles = (N + 15) / 16, nchunk = (K + 63) / 64;
  int s = (target + tiles - 1) / tiles;
  s = std::min(s, std::max(1, nchunk / minchunk));
  return std::max(1, std::min(8, s));
}

// split-K factor for a tiled GEMM whose output grid alone cannot fill 256 CUs (e.g. M = 386, N = 3584: 196 tiles)
int gemm_tiled_num_splits(int M, int N, int K, bool packed_bf16) {
  const long tiles = (long)((M + 63) / 64) * ((N + 127) / 128);
  // More than one chunk's rows on a long K (bf16 weights): the split count whose best tile (split_score against 1.25 PFLOP/s) plus the slabs' way
  // to memory and back is shortest, and only if that saves a tenth.  Product and consumer together, us, without / with: 1000 x 3584, K 22528 240 / 170
  // (three splits instead of 128 x 128 tiles); 600 x 3584, K 18944 107 (three) / 94; 2104 x 1536, K 10496 86 / 73; 1000 x 1536, K 8960 52 / 40.
  if (packed_bf16 && M > 448 && M <= 4096 && K >= 6144 && (K & 63) == 0 && (N & 15) == 0 && g_gemm_variant == 2) {
    GemmArgs a; a.M = M; a.N = N; a.K = K; a.w_packed = 1; a.lda = K;
    int best = 1;
    float best_us = 0.f;
    for (int S = 1; S <= 6; ++S) {
      const float us = 2e-9f * (float)M * (float)N * (float)K / (1.25f * split_score(a, S)) + (S > 1 ? (float)S * (float)M * (float)N * 8e-6f / 4.5f : 0.f);
      if (S == 1 || us < (best == 1 ? 0.9f : 1.f) * best_us) { best = S; best_us = us; }
    }
    return best;
  }
  if (tiles >= 400 || M > 4096) return 1;
  int s = (int)((640 + tiles - 1) / tiles);
  s = std::min(s, std::max(1, ((K + 63) / 64) / 8));
  s = std::max(1, std::min(4, s));
  // small variable-height tiles (bf16 weights): floor(F / 8) row tiles x 256-column tiles -> as many splits as fill one round of the chip
  // (7B chunk, M = 386: o / down 3 x 14 tiles x 6 = 252 blocks, q|k|v 3 x 18 x 4 = 216), never fewer than the 128-row rule gives
  if (packed_bf16 && vh_small_on() && vh_small_shape(M, K) && (N & 15) == 0) {
    const long vt = (long)(((M + 15) >> 4) >> 3) * ((N + 255) / 256);
    int sv = (int)std::min<long>(6, 256 / std::max<long>(1, vt));
    sv = std::min(sv, std::max(1, ((K + 63) / 64) / 8));
    s = std::max(s, sv);
  }
  return s;
}

static int gemm_w8(const GemmArgs& a, hipStream_t st) {
  if ((a.K & 63) || (a.N & 15) || (a.lda & 7) || a.wscale == nullptr) return LCC_ERR_SHAPE;
  if ((((uintptr_t)a.A | (uintptr_t)a.W) & 15) != 0 || ((uintptr_t)a.wscale & 15) != 0) return LCC_ERR_ALIGN;
  if (a.epilogue == EPI_SWIGLU && (a.N & 31)) return LCC_ERR_SHAPE;
  const uint8_t* W8 = reinterpret_cast<const uint8_t*>(a.W);
  const bool skinny = a.M <= 16 && a.epilogue != EPI_QUICK_GELU && a.epilogue != EPI_GELU_ERF && a.epilogue != EPI_RESIDUAL;
  if (skinny) {
    const int nchunk = a.K / 64;
    if (a.epilogue == EPI_SWIGLU) {
      gemv_w8_kernel<2, 2><<<dim3((a.N + 31) / 32, 1), dim3(256), 0, st>>>(a.A, a.lda, W8, a.wscale, nullptr, a.C, a.ldc, a.M, a.N, a.K, nchunk);
    } else if (a.partial != nullptr) {
      const int S = a.nsplit > 0 ? a.nsplit : 1;
      if (S > nchunk || a.tail.kind != 0) return LCC_ERR_ARG;
      gemv_w8_kernel<1, 0><<<dim3((a.N + 15) / 16, S), dim3(256), 0, st>>>(a.A, a.lda, W8, a.wscale, nullptr, a.partial, a.N, a.M, a.N, a.K,
                                                                             (nchunk + S - 1) / S);
    } else {
      gemv_w8_kernel<1, 1><<<dim3((a.N + 15) / 16, 1), dim3(256), 0, st>>>(a.A, a.lda, W8, a.wscale, a.bias, a.C, a.ldc, a.M, a.N, a.K, nchunk);
    }
    return 0;
  }
  // the tile kernels consume the fp8 fragments directly (e4m3 -> bf16 after the LDS read); forced variants without such a kernel take the 64 x 128 tile
  GemmArgs c = a; c.w_packed = 1;
  const bool part = a.partial != nullptr;
  if (part && (a.epilogue != EPI_NONE || a.nsplit < 1 || a.nsplit > 8 || a.nsplit > a.K / 64)) return LCC_ERR_ARG;
  if (a.epilogue == EPI_RESIDUAL && a.residual == nullptr) return LCC_ERR_ARG;
  // A C that gemm_bf16 refuses (8-byte stores would not be aligned) only ever went to the 256-column tiles, where they scored above a narrow tile
  // behind a dequantising pass: they take it by the same lines, and the other shapes refuse it.
  const bool odd = (a.ldc & 3) != 0 || ((uintptr_t)a.C & 15) != 0;
  const bool tall = !part && !odd && tall_wanted(c);
  const int big = (g_gemm_variant == 7) ? 0 : big_tile_rows(c, part ? a.nsplit : 1, odd);
  if (odd && big != 256 && big != 128) return (a.ldc & 3) != 0 ? LCC_ERR_SHAPE : LCC_ERR_ALIGN;
#define LCC_W8_TILE(EPI) (big == 256 ? launch_big<256, EPI>(c, st) : big == 192 ? launch_big<192, EPI>(c, st) : big == 160 ? launch_big<160, EPI>(c, st) : big == 128 ? launch_big<128, EPI>(c, st) : big == 129 ? launch_mid<EPI>(c, st) : launch_mid64<EPI>(c, st))
#define LCC_W8(EPI) (tall ? launch_tall<EPI>(c, st) : LCC_W8_TILE(EPI))
  if (part) { LCC_W8_TILE(EPI_PARTIAL); return 0; }
  switch (a.epilogue) {
    case EPI_NONE: LCC_W8(EPI_NONE); return 0;
    case EPI_QUICK_GELU: LCC_W8(EPI_QUICK_GELU); return 0;
    case EPI_GELU_ERF: LCC_W8(EPI_GELU_ERF); return 0;
    case EPI_RESIDUAL: LCC_W8(EPI_RESIDUAL); return 0;
    case EPI_SWIGLU: LCC_W8(EPI_SWIGLU); return 0;
    default: return LCC_ERR_ARG;
  }
#undef LCC_W8
#undef LCC_W8_TILE
}

int gemm_bf16(const GemmArgs& a, hipStream_t st) {
  if (a.M <= 0 || a.N <= 0 || a.K <= 0) return 0;
  if (a.w_fp8) return gemm_w8(a, st);
  if ((a.K & 7) || (a.N & 15) || (a.lda & 7) || (!a.w_packed && (a.ldw & 7)) || (a.ldc & 3)) return LCC_ERR_SHAPE;
  if ((((uintptr_t)a.A | (uintptr_t)a.W | (uintptr_t)a.C) & 15) != 0) return LCC_ERR_ALIGN;
  if (a.epilogue == EPI_SWIGLU && (a.N & 31)) return LCC_ERR_SHAPE;
  if (a.epilogue == EPI_RESIDUAL && a.residual == nullptr) return LCC_ERR_ARG;
  if (a.epilogue == EPI_VIT_QKV || a.epilogue == EPI_VIT_QK || a.epilogue == EPI_VIT_V) {
    // vision-tower q|k|v projection with RoPE / the V transpose in the epilogue: all three in one launch (E % 128 == 0), or q|k and V apart
    const VitQkvEpi& q = a.vq;
    const bool all = a.epilogue == EPI_VIT_QKV, qk = all || a.epilogue == EPI_VIT_QK, v = all || a.epilogue == EPI_VIT_V;
    if (!a.w_packed || a.partial != nullptr || !gemm_vit_qkv_eligible(a.M, q.E, a.K) || a.N != (all ? 3 : qk ? 2 : 1) * q.E || (all && (q.E & 127))) return LCC_ERR_ARG;
    if (qk && (q.cs == nullptr || q.sn == nullptr || a.C == nullptr)) return LCC_ERR_ARG;
    if (v && (q.grp_off == nullptr || q.vt == nullptr || q.total_blocks <= 0)) return LCC_ERR_ARG;
    if (qk && (((uintptr_t)q.cs | (uintptr_t)q.sn) & 15) != 0) return LCC_ERR_ALIGN;
    if ((v && ((uintptr_t)q.vt & 7) != 0) || (a.bias != nullptr && ((uintptr_t)a.bias & 7) != 0)) return LCC_ERR_ALIGN;
    if (!walk_offsets_fit(a)) return LCC_ERR_SHAPE;      // lda is E, whose square of weights is in memory
    g_launch_counts[LC_GEMM_VIT_QKV]++;
    int big = big_tile_rows(a, 1);
    if (big == 160) big = 192;
    if (big == 272) big = 256;      // the rotation / transposed-V epilogues live on the fixed-height 256-column tiles (129, 0: the 128-row one, or for q, k and V together the 128-column tiles)
    // The narrow tiles where a product without these epilogues takes them (up to 1,024 patches at 1,280 channels).  A tower of 32 blocks, us, 128 x 256 tiles / here: 140 patches
    // 2681 / 2370, 320 2896 / 2522, 560 3204 / 3004, 720 3387 / 3165, 880 3739 / 3501.  Under a cap on the workgroups only while their tiles all run at once: a unit gets less done with them
    // (128 units: 140 patches, 90 tiles, 3004 / 2617; 560, 270 tiles, 3842 / 3983; 768, 360, 4014 / 4238; 40 units: 560 8337 / 8623)
    const long tiles = (long)(big == 129 ? (a.M + 127) / 128 : (a.M + 63) / 64) * ((a.N + 127) / 128);
    const bool narrow = all && (big == 129 || big == 0) && (get_grid_cap() <= 0 || tiles <= get_grid_cap());
    if (narrow) {
      g_launch_counts[LC_GEMM_VIT_QKV_NARROW]++;
      big == 129 ? launch_mid_w<EPI_VIT_QKV, false>(a, st) : launch_strip_w<EPI_VIT_QKV, false>(a, st);
    } else if (all) launch_vit<EPI_VIT_QKV>(a, big, st);
    else if (qk) launch_vit<EPI_VIT_QK>(a, big, st);
    else launch_vit<EPI_VIT_V>(a, big, st);
    return 0;
  }
  // weight-streaming path: up to g_skinny_rows rows (64: decode batches of 17-64 streams multiply every weight fragment with 2-4 activation
  // fragments; lcc_debug_set_skinny_rows(16) restores the round-3 routing of 17-64 rows through the 64-row GEMM tiles)
  // (a forced GEMM tile variant -- tests, A/B runs -- keeps 17-64 rows on the tiles it asks for)
  const bool skinny = gemm_routes_skinny(a.M, a.K, false) && a.epilogue != EPI_QUICK_GELU && a.epilogue != EPI_GELU_ERF && a.epilogue != EPI_RESIDUAL;
  if (skinny) {
    const int nchunk = (a.K + 63) / 64;
    if (a.epilogue == EPI_SWIGLU) {
      launch_gemv_rows<2>(a, 1, a.C, a.ldc, nchunk, st);
    } else if (a.partial != nullptr) {
      const int S = a.nsplit > 0 ? a.nsplit : 1;
      if (S > nchunk) return LCC_ERR_SHAPE;
      if (a.tail.kind != 0) {   // fused tail: last-arriving block reduces the slabs and runs the consumer (M <= 2, packed W)
        if (a.M > 2 || !a.w_packed || a.tail.counter == nullptr || S > 8 || (a.tail.kind == 1 && (a.N > 8192 || (a.N & 7)))) return LCC_ERR_ARG;
        g_launch_counts[LC_GEMV_FUSED_TAIL]++;
        gemv_skinny_kernel<1, 3, true, 1, 1><<<dim3((a.N + 15) / 16, S), dim3(256), 0, st>>>(
            a.A, a.lda, a.W, a.ldw, nullptr, a.partial, a.N, a.M, a.N, a.K, (nchunk + S - 1) / S, a.tail);
        return 0;
      }
      launch_gemv_rows<0>(a, S, a.partial, a.N, (nchunk + S - 1) / S, st);
    } else {
      launch_gemv_rows<1>(a, 1, a.C, a.ldc, nchunk, st);
    }
    return 0;
  }
  if (a.partial != nullptr) {   // split-K slabs on the tiled path (prefill GEMMs with few output tiles)
    if (a.epilogue != EPI_NONE || a.nsplit < 1 || a.nsplit > 8 || a.nsplit > (a.K + 63) / 64) return LCC_ERR_ARG;
    const int big = big_tile_rows(a, a.nsplit);
    if (big == 272) launch_vh<EPI_PARTIAL>(a, st);
    else if (big == 144) launch_vh_small(a, st);
    else if (big == 256) launch_big<256, EPI_PARTIAL>(a, st);
    else if (big == 192) launch_big<192, EPI_PARTIAL>(a, st);
    else if (big == 160) launch_big<160, EPI_PARTIAL>(a, st);
    else if (big == 128) launch_big<128, EPI_PARTIAL>(a, st);
    else if (big == 129) launch_mid<EPI_PARTIAL>(a, st);
    else launch_tiled<64, EPI_PARTIAL>(a, st);
    return 0;
  }
  switch (a.epilogue) {
    case EPI_NONE: launch_tiled_bm<EPI_NONE>(a, st); break;
    case EPI_QUICK_GELU: launch_tiled_bm<EPI_QUICK_GELU>(a, st); break;
    case EPI_GELU_ERF: launch_tiled_bm<EPI_GELU_ERF>(a, st); break;
    case EPI_RESIDUAL: launch_tiled_bm<EPI_RESIDUAL>(a, st); break;
    case EPI_SWIGLU: launch_tiled_bm<EPI_SWIGLU>(a, st); break;
    default: return LCC_ERR_ARG;
  }
  return 0;
}

}  // namespace lcc
