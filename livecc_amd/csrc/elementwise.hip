// HBM-bound elementwise / normalisation / layout kernels of the LiveCC hot path (gfx950).
// All bf16 traffic is 16 bytes per lane; reductions are wave shuffles (64 lanes) + a tiny LDS step.
// Every kernel reproduces the rounding points of the HF op it replaces (cited per kernel).
#include "common.h"
#include "kernels.h"

namespace lcc {

static inline int64_t host_min(int64_t a, int64_t b) { return a < b ? a : b; }

// ------------------------------------------------------------------------------------------------
// K1: rescale + normalise + patchify, uint8 frames -> bf16 patch rows [P, 1176]
//   HF video_processing_qwen2_vl.py:236-274 (patch order t, h/2, w/2, 2, 2; feature c*392+tt*196+py*14+px)
//   HF image_processing_backends.py:307-333: (float(x) - mean*255) / (std*255) in fp32, then the model casts
//   pixel_values to bf16 (modeling_qwen2_vl.py:1044).  The reference ships 4704 B/patch of fp32 over PCIe;
//   here 1176 B/patch of uint8 are read from HBM.
// layout 0: [T,H,W,3] (decoder-native), 1: [T,3,H,W] (what get_smart_resized_clip returns)
// ------------------------------------------------------------------------------------------------
struct NormConst { float mean[3], stdv[3]; };

__global__ __launch_bounds__(256) void patchify_norm_kernel(const uint8_t* __restrict__ f, int layout, int T, int H,
                                                            int W, bf16_t* __restrict__ out, int ld, NormConst nc,
                                                            int P, int chunks_per_row) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= P * chunks_per_row) return;
  const int p = idx / chunks_per_row, c8 = (idx - p * chunks_per_row) * 8;
  const int gh = H / 14, gw = W / 14, hb_n = gh / 2, wb_n = gw / 2;
  int r = p;
  const int mw = r & 1; r >>= 1;
  const int mh = r & 1; r >>= 1;
  const int wb = r % wb_n; r /= wb_n;
  const int hb = r % hb_n; r /= hb_n;
  const int tg = r;
  const int py0 = (hb * 2 + mh) * 14, px0 = (wb * 2 + mw) * 14;
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    int col = c8 + e;
    const int c = col / 392; col -= c * 392;
    const int tt = col / 196; col -= tt * 196;
    const int py = col / 14, px = col - py * 14;
    const int t = min(tg * 2 + tt, T - 1);  // odd T: last frame repeated (video_processing_qwen2_vl.py:246-250)
    const int y = py0 + py, x = px0 + px;
    const size_t a = layout == 0 ? (((size_t)t * H + y) * W + x) * 3 + c : (((size_t)t * 3 + c) * H + y) * W + x;
    v[e] = ((float)f[a] - nc.mean[c]) / nc.stdv[c];
  }
  st16(out + (size_t)p * ld + c8, (u32x4){pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])});
}

int patchify_norm_u8(const uint8_t* frames, int layout, int T, int H, int W, const float* mean255,
                     const float* std255, bf16_t* out, int ld, hipStream_t st) {
  if (H % 28 || W % 28 || T <= 0 || (ld & 7) || ld < 1176) return LCC_ERR_SHAPE;
  const int P = ((T + 1) / 2) * (H / 14) * (W / 14);
  NormConst nc;
  for (int i = 0; i < 3; ++i) { nc.mean[i] = mean255[i]; nc.stdv[i] = std255[i]; }
  const int cpr = 1176 / 8;
  patchify_norm_kernel<<<dim3((P * cpr + 255) / 256), dim3(256), 0, st>>>(frames, layout, T, H, W, out, ld, nc, P, cpr);
  return 0;
}

__global__ __launch_bounds__(256) void cast_f32_bf16_kernel(const float* __restrict__ in, bf16_t* __restrict__ out,
                                                            int64_t n8) {
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(in + i * 8), b = *reinterpret_cast<const f32x4*>(in + i * 8 + 4);
    st16(out + i * 8, (u32x4){pack2(a[0], a[1]), pack2(a[2], a[3]), pack2(b[0], b[1]), pack2(b[2], b[3])});
  }
}
int cast_f32_bf16(const float* in, bf16_t* out, int64_t n, hipStream_t st) {
  if (n & 7) return LCC_ERR_SHAPE;
  const int64_t n8 = n / 8;
  if (n8 == 0) return 0;
  cast_f32_bf16_kernel<<<dim3((unsigned)host_min((n8 + 255) / 256, 4096)), dim3(256), 0, st>>>(in, out, n8);
  return 0;
}

// ------------------------------------------------------------------------------------------------
// row kernels: NW waves cooperate on one row of `dim` elements, MAXC 8-element chunks per thread in registers
// ------------------------------------------------------------------------------------------------
// LayerNorm (ViT): torch native_layer_norm on bf16 = fp32 statistics, y = (x-mean)*rstd*w + b, one rounding.
// HF modeling_qwen2_vl.py:428-429 (norm1/norm2), 281 (merger ln_q); eps 1e-6.
template <int NW, int MAXC>
__global__ __launch_bounds__(NW * 64) void layernorm_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                            const bf16_t* __restrict__ b, bf16_t* __restrict__ y,
                                                            int dim, float eps) {
  __shared__ float red[NW];
  const int row = blockIdx.x, tid = threadIdx.x, nchunk = dim / 8;
  const bf16_t* xr = x + (size_t)row * dim;
  // the row, the weights and the biases are asked for at once, at clamped addresses: behind branches a row of 1,280 was three trips to memory in a row and the
  // weights a fourth (in a row of launches: 1,456 rows 4.1 -> 3.6 us, 15,840 rows 15.6 -> 14.0)
  u32x4 xq[MAXC], wq[MAXC], bq[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) xq[c] = ld16(xr + min(tid + c * NW * 64, nchunk - 1) * 8);
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int at = min(tid + c * NW * 64, nchunk - 1) * 8;
    wq[c] = ld16(w + at); bq[c] = ld16(b + at);
  }
  float v[MAXC][8];
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[c][2 * e] = lo2f(xq[c][e]); v[c][2 * e + 1] = hi2f(xq[c][e]); }
    if (tid + c * NW * 64 < nchunk) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[c][e];
    }
  }
  const float mean = block_sum<NW>(s, red) / (float)dim;
  float s2 = 0.f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = tid + c * NW * 64;
    if (ch < nchunk) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = v[c][e] - mean; s2 += d * d; }
    }
  }
  const float var = block_sum<NW>(s2, red) / (float)dim;
  const float rstd = rsqrtf(var + eps);
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = tid + c * NW * 64;
    if (ch < nchunk) {
      float o[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] = (v[c][2 * e] - mean) * rstd * lo2f(wq[c][e]) + lo2f(bq[c][e]);
        o[2 * e + 1] = (v[c][2 * e + 1] - mean) * rstd * hi2f(wq[c][e]) + hi2f(bq[c][e]);
      }
      st16(y + (size_t)row * dim + ch * 8,
           (u32x4){pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7])});
    }
  }
}

int layernorm_bf16(const bf16_t* x, const bf16_t* w, const bf16_t* b, bf16_t* y, int rows, int dim, float eps,
                   hipStream_t st) {
  if (rows <= 0) return 0;
  if ((dim & 7) || dim > 4 * 64 * 8 * 4) return LCC_ERR_SHAPE;
  if (dim <= 0) return 0;          // the kernel's loads are clamped to a row's last piece
  if (dim <= 64 * 8 * 2) layernorm_kernel<1, 2><<<dim3(rows), dim3(64), 0, st>>>(x, w, b, y, dim, eps);
  else if (dim <= 64 * 8 * 3) layernorm_kernel<1, 3><<<dim3(rows), dim3(64), 0, st>>>(x, w, b, y, dim, eps);
  else if (dim <= 64 * 8 * 4) layernorm_kernel<1, 4><<<dim3(rows), dim3(64), 0, st>>>(x, w, b, y, dim, eps);
  else layernorm_kernel<4, 4><<<dim3(rows), dim3(256), 0, st>>>(x, w, b, y, dim, eps);
  return 0;
}

// (residual add +) RMSNorm (LLM).  HF modeling_qwen2_vl.py:96-110: fp32 x, var = mean(x^2),
// xhat = x*rsqrt(var+eps) -> cast to bf16 -> weight * xhat (bf16 product, rounded).  Residual add =
// `residual + hidden_states` on bf16 tensors (decoder layer 604, 610): fp32 add, one rounding.
// DELTA 0: none; 1: bf16 delta [rows,dim]; 2: fp32 split-K slabs [nsplit][rows][dim] (summed in slab order,
// rounded to bf16 like the Linear output they stand for).
template <int NW, int MAXC, int DELTA, int NS>
__global__ __launch_bounds__(NW * 64) void add_rmsnorm_kernel(bf16_t* __restrict__ h, const bf16_t* __restrict__ dbf,
                                                              const float* __restrict__ dpart, int nsplit, int rows,
                                                              const bf16_t* __restrict__ w, bf16_t* __restrict__ y,
                                                              int dim, float eps) {
  __shared__ float red[NW];
  const int row = blockIdx.x, tid = threadIdx.x, nchunk = dim / 8;
  bf16_t* hr = h + (size_t)row * dim;
  float v[MAXC][8];
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = tid + c * NW * 64;
    if (ch < nchunk) {
      const u32x4 q = ld16(hr + ch * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) { v[c][2 * e] = lo2f(q[e]); v[c][2 * e + 1] = hi2f(q[e]); }
      if (DELTA == 1) {
        const u32x4 d = ld16(dbf + (size_t)row * dim + ch * 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[c][2 * e] = rbf(v[c][2 * e] + lo2f(d[e])); v[c][2 * e + 1] = rbf(v[c][2 * e + 1] + hi2f(d[e])); }
      } else if (DELTA == 2) {
        float d[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        f32x4 pa[NS], pb[NS];  // NS is a compile-time slab count: straight-line loads, one L2/MALL round trip
#pragma unroll
        for (int sp = 0; sp < NS; ++sp) {
          const float* pp = dpart + ((size_t)sp * rows + row) * dim + ch * 8;
          pa[sp] = *reinterpret_cast<const f32x4*>(pp); pb[sp] = *reinterpret_cast<const f32x4*>(pp + 4);
        }
#pragma unroll
        for (int sp = 0; sp < NS; ++sp)   // slab order
#pragma unroll
          for (int e = 0; e < 4; ++e) { d[e] += pa[sp][e]; d[4 + e] += pb[sp][e]; }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[c][e] = rbf(v[c][e] + rbf(d[e]));
      }
      if (DELTA != 0)
        st16(hr + ch * 8, (u32x4){pack2(v[c][0], v[c][1]), pack2(v[c][2], v[c][3]), pack2(v[c][4], v[c][5]),
                                  pack2(v[c][6], v[c][7])});
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[c][e] * v[c][e];
    }
  }
  if (w == nullptr) return;
  const float var = block_sum<NW>(s, red) / (float)dim;
  const float rstd = rsqrtf(var + eps);
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = tid + c * NW * 64;
    if (ch < nchunk) {
      const u32x4 wq = ld16(w + ch * 8);
      float o[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] = lo2f(wq[e]) * rbf(v[c][2 * e] * rstd);
        o[2 * e + 1] = hi2f(wq[e]) * rbf(v[c][2 * e + 1] * rstd);
      }
      st16(y + (size_t)row * dim + ch * 8,
           (u32x4){pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7])});
    }
  }
}

int add_rmsnorm_bf16(bf16_t* h, const bf16_t* delta_bf16, const float* delta_partial, int nsplit, const bf16_t* w,
                     bf16_t* y, int rows, int dim, float eps, hipStream_t st) {
  if (rows <= 0) return 0;
  if ((dim & 7) || dim > 4 * 64 * 8 * 4) return LCC_ERR_SHAPE;
  if (delta_bf16 != nullptr && delta_partial != nullptr) return LCC_ERR_ARG;
  if (delta_partial != nullptr && (nsplit < 1 || nsplit > 8)) return LCC_ERR_SHAPE;
  if (delta_partial != nullptr) {
#define LCC_ADDN(NS) add_rmsnorm_kernel<4, 4, 2, NS><<<dim3(rows), dim3(256), 0, st>>>(h, nullptr, delta_partial, nsplit, rows, w, y, dim, eps)
    switch (nsplit) {
      case 1: LCC_ADDN(1); break; case 2: LCC_ADDN(2); break; case 3: LCC_ADDN(3); break; case 4: LCC_ADDN(4); break;
      case 5: LCC_ADDN(5); break; case 6: LCC_ADDN(6); break; case 7: LCC_ADDN(7); break; default: LCC_ADDN(8); break;
    }
#undef LCC_ADDN
  } else if (delta_bf16 != nullptr)
    add_rmsnorm_kernel<4, 4, 1, 1><<<dim3(rows), dim3(256), 0, st>>>(h, delta_bf16, nullptr, 0, rows, w, y, dim, eps);
  else
    add_rmsnorm_kernel<4, 4, 0, 1><<<dim3(rows), dim3(256), 0, st>>>(h, nullptr, nullptr, 0, rows, w, y, dim, eps);
  return 0;
}

int rmsnorm_bf16(const bf16_t* x, const bf16_t* w, bf16_t* y, int rows, int dim, float eps, hipStream_t st) {
  if (w == nullptr) return LCC_ERR_ARG;
  return add_rmsnorm_bf16(const_cast<bf16_t*>(x), nullptr, nullptr, 0, w, y, rows, dim, eps, st);
}

// ------------------------------------------------------------------------------------------------
// ViT 2-D RoPE on q,k (in place in the qkv GEMM output) + V written blocked-transposed for the attention
// kernel.  HF modeling_qwen2_vl.py:225-248: fp32 q*cos + rotate_half(q)*sin, one rounding to bf16; head_dim
// 80 = cat(freqs, freqs) with freqs = [20 h-freqs | 20 w-freqs] (700-713, vision_utils.py:81-127).
// cos/sin: fp32 [P, 40].  One thread = 8 channels (c..c+7, c < 40) and their partners (c+40..): 5 threads per
// (patch, head, q|k), plus 10 threads per (patch, head) moving V.
// vt layout: [head][block][80][32], block = seg_blk_start[seg] + local_index/32.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void vit_rope_vt_kernel(bf16_t* __restrict__ qkv, const float* __restrict__ cs,
                                                          const float* __restrict__ sn,
                                                          const int32_t* __restrict__ seg_of_patch,
                                                          const int32_t* __restrict__ seg_start,
                                                          const int32_t* __restrict__ seg_blk_start,
                                                          bf16_t* __restrict__ vt, int P, int heads, int total_blocks) {
  constexpr int D = 80, HALF = 40;
  const int E = heads * D;
  const int64_t n_rope = (int64_t)P * heads * 10;                // 5 chunks x (q, k) per (patch, head)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx < n_rope) {
    const int it = (int)(idx % 10);
    const int64_t ph = idx / 10;
    const int h = (int)(ph % heads), p = (int)(ph / heads);
    const int which = it / 5, c0 = (it % 5) * 8;
    bf16_t* base = qkv + (size_t)p * 3 * E + which * E + h * D;
    const u32x4 a = ld16(base + c0), b = ld16(base + c0 + HALF);
    float x1[8], x2[8], o1[8], o2[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) { x1[2 * e] = lo2f(a[e]); x1[2 * e + 1] = hi2f(a[e]); x2[2 * e] = lo2f(b[e]); x2[2 * e + 1] = hi2f(b[e]); }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float c = cs[(size_t)p * HALF + c0 + e], s = sn[(size_t)p * HALF + c0 + e];
      vit_rope_pair(x1[e], x2[e], c, s, o1[e], o2[e]);  // q*cos + rotate_half(q)*sin, products rounded separately as in HF
    }
    st16(base + c0, (u32x4){pack2(o1[0], o1[1]), pack2(o1[2], o1[3]), pack2(o1[4], o1[5]), pack2(o1[6], o1[7])});
    st16(base + c0 + HALF, (u32x4){pack2(o2[0], o2[1]), pack2(o2[2], o2[3]), pack2(o2[4], o2[5]), pack2(o2[6], o2[7])});
    return;
  }
  // V -> blocked-transposed [head][block][80][32].  One thread = 8 consecutive patches x 8 channels: eight 16-byte row loads
  // (coalesced across the lanes of a patch row), an 8x8 transpose in registers, eight 16-byte stores of 8 consecutive keys each.
  // (The first version stored every element with its own 2-byte store: 141 us for 11648 patches, ~8x the HBM time.)
  const int64_t j = idx - n_rope;
  const int n_grp = (P + 7) / 8;
  if (j >= (int64_t)n_grp * heads * 10) return;
  const int c0 = (int)(j % 10) * 8;
  const int64_t gh = j / 10;
  const int h = (int)(gh % heads), p0 = (int)(gh / heads) * 8;
  const int sg = seg_of_patch[p0];
  const int kl0 = p0 - seg_start[sg];
  const bool aligned = (p0 + 7 < P) && (seg_of_patch[min(p0 + 7, P - 1)] == sg) && ((kl0 & 7) == 0);
  if (aligned) {
    u32x4 a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = ld16(qkv + (size_t)(p0 + k) * 3 * E + 2 * E + h * D + c0);
    bf16_t* dst = vt + (((size_t)h * total_blocks + seg_blk_start[sg] + (kl0 >> 5)) * D + c0) * 32 + (kl0 & 31);
#pragma unroll
    for (int dd = 0; dd < 8; ++dd) {               // channel c0 + dd: its 8 keys
      unsigned v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (dd & 1) ? (a[k][dd >> 1] >> 16) : (a[k][dd >> 1] & 0xffffu);
      st16(dst + dd * 32, (u32x4){v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)});
    }
    return;
  }
  for (int k = 0; k < 8 && p0 + k < P; ++k) {      // ragged group (segment length not a multiple of 8): element stores
    const int p = p0 + k, s2 = seg_of_patch[p], kl = p - seg_start[s2];
    const u32x4 a = ld16(qkv + (size_t)p * 3 * E + 2 * E + h * D + c0);
    bf16_t* dst = vt + (((size_t)h * total_blocks + seg_blk_start[s2] + (kl >> 5)) * D + c0) * 32 + (kl & 31);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dst[(2 * e) * 32] = (bf16_t)(a[e] & 0xffffu);
      dst[(2 * e + 1) * 32] = (bf16_t)(a[e] >> 16);
    }
  }
}

int vit_rope_vt_bf16(bf16_t* qkv, const float* cos, const float* sin, const int32_t* seg_of_patch,
                     const int32_t* seg_start, const int32_t* seg_blk_start, bf16_t* vt, int P, int heads,
                     int total_blocks, hipStream_t st) {
  if (P <= 0) return 0;
  const int64_t n = (int64_t)P * heads * 10 + (int64_t)((P + 7) / 8) * heads * 10;
  vit_rope_vt_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(qkv, cos, sin, seg_of_patch, seg_start,
                                                                             seg_blk_start, vt, P, heads, total_blocks);
  return 0;
}

// ------------------------------------------------------------------------------------------------
// M-RoPE cos/sin tables: HF modeling_qwen2_vl.py:156-169: freqs = inv_freq * pos (fp32), cos/sin in fp32,
// cast to the model dtype (bf16).  Only the 64 unique channels are stored ([S,64]); channel c takes the
// position axis mrope_section assigns to it (180-222: [16,24,24] -> t,h,w).
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void mrope_table_kernel(const int32_t* __restrict__ pos3, const float* __restrict__ inv_freq,
                                                          int S, int sec_t, int sec_h, bf16_t* __restrict__ cs,
                                                          bf16_t* __restrict__ sn) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= S * 64) return;
  const int s = idx >> 6, c = idx & 63;
  const int axis = c < sec_t ? 0 : (c < sec_t + sec_h ? 1 : 2);
  const float ang = inv_freq[c] * (float)pos3[(size_t)axis * S + s];
  cs[idx] = f2bf(cosf(ang));
  sn[idx] = f2bf(sinf(ang));
}

int mrope_table(const int32_t* pos3, const float* inv_freq, int S, int sec_t, int sec_h, bf16_t* cos, bf16_t* sin,
                hipStream_t st) {
  if (S <= 0) return 0;
  mrope_table_kernel<<<dim3((S * 64 + 255) / 256), dim3(256), 0, st>>>(pos3, inv_freq, S, sec_t, sec_h, cos, sin);
  return 0;
}

// decode variant: one position per stream taken from a device counter (all three axes equal:
// HF modeling_qwen2_vl.py:1349-1351), so that consecutive decode steps need no host round trip.
__global__ __launch_bounds__(64) void mrope_table_decode_kernel(const int32_t* __restrict__ slots, const int32_t* __restrict__ pos,
                                                                const float* __restrict__ inv_freq,
                                                                bf16_t* __restrict__ cs, bf16_t* __restrict__ sn) {
  const int b = blockIdx.x, c = threadIdx.x;
  const float ang = inv_freq[c] * (float)pos[slots[b]];
  cs[b * 64 + c] = f2bf(cosf(ang));
  sn[b * 64 + c] = f2bf(sinf(ang));
}
int mrope_table_decode(const int32_t* slots, const int32_t* pos, const float* inv_freq, int B, bf16_t* cos, bf16_t* sin,
                       hipStream_t st) {
  if (B <= 0) return 0;
  mrope_table_decode_kernel<<<dim3(B), dim3(64), 0, st>>>(slots, pos, inv_freq, cos, sin);
  return 0;
}

// ------------------------------------------------------------------------------------------------
// M-RoPE apply + in-place KV append (replaces apply_multimodal_rotary_pos_emb 180-222 and
// DynamicLayer.update's torch.cat, cache_utils.py:127-146: 57,344 B/token written instead of 2*L*57,344 moved).
// bf16 op-by-op rounding as HF: out = bf16(bf16(x*cos) + bf16(rot(x)*sin)).
// K -> cache [Hkv][Lmax][128]; V -> cache blocked-transposed [Hkv][Lmax/32][128][32]; q -> q_out [S, Hq*128].
// One thread = 8 channels c..c+7 (c < 64) and partners c+64: 8 threads per rope head; 16 threads per V head.
// QSRC 0: qkv bf16 [S, ld]; 1: fp32 split-K slabs [nsplit][S][ld] + bias (decode path).
// ------------------------------------------------------------------------------------------------
template <int QSRC, int NS>
LCC_DEVICE void load8(const bf16_t* qkv, const float* part, int S, const bf16_t* bias, int s, int ld,
                      int col, float (&v)[8]) {
  if (QSRC == 0) {
    const u32x4 a = ld16(qkv + (size_t)s * ld + col);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[2 * e] = lo2f(a[e]); v[2 * e + 1] = hi2f(a[e]); }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    f32x4 pa[NS], pb[NS];
#pragma unroll
    for (int sp = 0; sp < NS; ++sp) {
      const float* pp = part + ((size_t)sp * S + s) * ld + col;
      pa[sp] = *reinterpret_cast<const f32x4*>(pp); pb[sp] = *reinterpret_cast<const f32x4*>(pp + 4);
    }
#pragma unroll
    for (int sp = 0; sp < NS; ++sp)
#pragma unroll
      for (int e = 0; e < 4; ++e) { v[e] += pa[sp][e]; v[4 + e] += pb[sp][e]; }
    const u32x4 bq = ld16(bias + col);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[2 * e] = rbf(v[2 * e] + lo2f(bq[e])); v[2 * e + 1] = rbf(v[2 * e + 1] + hi2f(bq[e])); }
  }
}

template <int QSRC, int NS>
__global__ __launch_bounds__(256) void rope_kv_append_kernel(
    const bf16_t* __restrict__ qkv, const float* __restrict__ part, const bf16_t* __restrict__ bias,
    const bf16_t* __restrict__ cs, const bf16_t* __restrict__ sn, const int32_t* __restrict__ tok_stream,
    const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ kv_len, bf16_t* const* __restrict__ kv_base,
    KvLayout lay, int layer, bf16_t* __restrict__ q_out, int S, int n_q_heads) {
  constexpr int D = 128;
  const int hkv = lay.n_kv_heads;
  const int per_tok = (n_q_heads + hkv) * 8 + hkv * 16;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)S * per_tok) return;
  const int s = (int)(idx / per_tok);
  int it = (int)(idx - (int64_t)s * per_tok);
  const int ld = (n_q_heads + 2 * hkv) * D;
  const int strm = tok_stream[s];
  const int slot = tok_pos != nullptr ? tok_pos[s] : kv_len[strm];  // cache index of this token
  bf16_t* base = kv_base[strm] + (size_t)layer * lay.layer_stride();
  if (it < (n_q_heads + hkv) * 8) {
    const int head = it >> 3, c0 = (it & 7) * 8;
    float x1[8], x2[8], o1[8], o2[8];
    load8<QSRC, NS>(qkv, part, S, bias, s, ld, head * D + c0, x1);
    load8<QSRC, NS>(qkv, part, S, bias, s, ld, head * D + c0 + 64, x2);
    const u32x4 cq = ld16(cs + (size_t)s * 64 + c0), sq = ld16(sn + (size_t)s * 64 + c0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float c = (e & 1) ? hi2f(cq[e >> 1]) : lo2f(cq[e >> 1]);
      const float sv = (e & 1) ? hi2f(sq[e >> 1]) : lo2f(sq[e >> 1]);
      o1[e] = rbf(x1[e] * c) + rbf(-x2[e] * sv);
      o2[e] = rbf(x2[e] * c) + rbf(x1[e] * sv);
    }
    const u32x4 r1 = (u32x4){pack2(o1[0], o1[1]), pack2(o1[2], o1[3]), pack2(o1[4], o1[5]), pack2(o1[6], o1[7])};
    const u32x4 r2 = (u32x4){pack2(o2[0], o2[1]), pack2(o2[2], o2[3]), pack2(o2[4], o2[5]), pack2(o2[6], o2[7])};
    bf16_t* dst;
    if (head < n_q_heads) dst = q_out + (size_t)s * n_q_heads * D + head * D;
    else dst = base + (size_t)(head - n_q_heads) * lay.head_stride() + (size_t)slot * D;
    st16(dst + c0, r1);
    st16(dst + c0 + 64, r2);
  } else {
    it -= (n_q_heads + hkv) * 8;
    const int hv = it >> 4, c0 = (it & 15) * 8;
    float x[8];
    load8<QSRC, NS>(qkv, part, S, bias, s, ld, (n_q_heads + hkv + hv) * D + c0, x);
    bf16_t* dst = base + lay.kv_stride() + (size_t)hv * lay.head_stride() + ((size_t)(slot >> 5) * D + c0) * 32 + (slot & 31);
#pragma unroll
    for (int e = 0; e < 8; ++e) dst[e * 32] = f2bf(x[e]);
  }
}

int rope_kv_append_bf16(const bf16_t* qkv_bf16, const float* qkv_partial, int nsplit, const bf16_t* bias,
                        const bf16_t* cos, const bf16_t* sin, const int32_t* tok_stream, const int32_t* tok_pos,
                        const int32_t* kv_len, bf16_t* const* kv_base, KvLayout lay, int layer, bf16_t* q_out, int S,
                        int n_q_heads, hipStream_t st) {
  if (S <= 0) return 0;
  if (lay.head_dim != 128 || (lay.lmax & 31)) return LCC_ERR_SHAPE;
  if (tok_pos == nullptr && kv_len == nullptr) return LCC_ERR_ARG;
  const int per_tok = (n_q_heads + lay.n_kv_heads) * 8 + lay.n_kv_heads * 16;
  const int64_t n = (int64_t)S * per_tok;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (qkv_partial != nullptr) {
    if (bias == nullptr) return LCC_ERR_ARG;
    if (nsplit < 1 || nsplit > 8) return LCC_ERR_SHAPE;
#define LCC_ROPEN(NS) rope_kv_append_kernel<1, NS><<<grid, dim3(256), 0, st>>>(nullptr, qkv_partial, bias, cos, sin, tok_stream, \
                                                               tok_pos, kv_len, kv_base, lay, layer, q_out, S, n_q_heads)
    switch (nsplit) {
      case 1: LCC_ROPEN(1); break; case 2: LCC_ROPEN(2); break; case 3: LCC_ROPEN(3); break; case 4: LCC_ROPEN(4); break;
      case 5: LCC_ROPEN(5); break; case 6: LCC_ROPEN(6); break; case 7: LCC_ROPEN(7); break; default: LCC_ROPEN(8); break;
    }
#undef LCC_ROPEN
  } else {
    rope_kv_append_kernel<0, 1><<<grid, dim3(256), 0, st>>>(qkv_bf16, nullptr, nullptr, cos, sin, tok_stream, tok_pos, kv_len,
                                                            kv_base, lay, layer, q_out, S, n_q_heads);
  }
  return 0;
}

// ------------------------------------------------------------------------------------------------
// token embedding gather + ViT row scatter (HF modeling_qwen2_vl.py:1159-1176: embed_tokens then
// masked_scatter of the video rows in order).  vit_index[s] < 0 -> embedding row ids[s]; else ViT row.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void embed_gather_kernel(const int32_t* __restrict__ ids, const int32_t* __restrict__ indirect,
                                                           const int32_t* __restrict__ vit_index,
                                                           const bf16_t* __restrict__ table, const bf16_t* __restrict__ vit_rows,
                                                           bf16_t* __restrict__ out, int S, int dim) {
  const int cpr = dim / 8;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < (int64_t)S * cpr; i += (int64_t)gridDim.x * 256) {
    const int s = (int)(i / cpr), c = (int)(i - (int64_t)s * cpr);
    const int vi = vit_index != nullptr ? vit_index[s] : -1;
    const int id = indirect != nullptr ? ids[indirect[s]] : ids[s];
    const bf16_t* src = vi >= 0 ? vit_rows + (size_t)vi * dim : table + (size_t)id * dim;
    st16(out + (size_t)s * dim + c * 8, ld16(src + c * 8));
  }
}
int embed_gather_bf16(const int32_t* ids, const int32_t* indirect, const int32_t* vit_index, const bf16_t* table,
                      const bf16_t* vit_rows, bf16_t* out, int S, int dim, hipStream_t st) {
  if (S <= 0) return 0;
  if (dim & 7) return LCC_ERR_SHAPE;
  const int64_t n = (int64_t)S * (dim / 8);
  embed_gather_kernel<<<dim3((unsigned)host_min((n + 255) / 256, 8192)), dim3(256), 0, st>>>(ids, indirect, vit_index, table, vit_rows, out, S, dim);
  return 0;
}

__global__ __launch_bounds__(256) void gather_rows_kernel(const bf16_t* __restrict__ in, const int32_t* __restrict__ rows,
                                                          bf16_t* __restrict__ out, int n, int dim) {
  const int cpr = dim / 8;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < (int64_t)n * cpr; i += (int64_t)gridDim.x * 256) {
    const int r = (int)(i / cpr), c = (int)(i - (int64_t)r * cpr);
    st16(out + (size_t)r * dim + c * 8, ld16(in + (size_t)rows[r] * dim + c * 8));
  }
}
int gather_rows_bf16(const bf16_t* in, const int32_t* rows, bf16_t* out, int n, int dim, hipStream_t st) {
  if (n <= 0) return 0;
  if (dim & 7) return LCC_ERR_SHAPE;
  const int64_t t = (int64_t)n * (dim / 8);
  gather_rows_kernel<<<dim3((unsigned)host_min((t + 255) / 256, 4096)), dim3(256), 0, st>>>(in, rows, out, n, dim);
  return 0;
}

// standalone SwiGLU for the HF plugin path (liger's LigerSwiGLUMLP slot): out = bf16(silu(g) * u)
__global__ __launch_bounds__(256) void swiglu_kernel(const bf16_t* __restrict__ g, const bf16_t* __restrict__ u,
                                                     bf16_t* __restrict__ out, int64_t n8) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const u32x4 a = ld16(g + i * 8), b = ld16(u + i * 8);
    float o[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[2 * e] = silu_bf16(lo2f(a[e])) * lo2f(b[e]);
      o[2 * e + 1] = silu_bf16(hi2f(a[e])) * hi2f(b[e]);
    }
    st16(out + i * 8, (u32x4){pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7])});
  }
}
int swiglu_bf16(const bf16_t* g, const bf16_t* u, bf16_t* out, int64_t n, hipStream_t st) {
  if (n & 7) return LCC_ERR_SHAPE;
  const int64_t n8 = n / 8;
  if (n8 == 0) return 0;
  swiglu_kernel<<<dim3((unsigned)host_min((n8 + 255) / 256, 8192)), dim3(256), 0, st>>>(g, u, out, n8);
  return 0;
}

// ------------------------------------------------------------------------------------------------
// bicubic antialias resize of uint8 frames (ref livecc_utils/video_process_patch.py:150-155 =
// torchvision.transforms.functional.resize(uint8, BICUBIC, antialias=True) = float32 ATen `_upsample_bicubic2d_aa` + clamp +
// round-half-even).  Separable, width pass then height pass, fp32, taps accumulated in order: t = s0*w0; t = fma(s_j, w_j, t)
// (ATen's `interpolate_aa_single_dim` as compiled: bit-identical results, tests/test_gpu_resize.py).  The tap tables come from
// the host (livecc_amd/resize.py) so that no weight is ever computed with different rounding on the device.
// HBM-bound byte work: pass 1 reads each source byte ~support times out of L2, writes Hin*Wout floats; pass 2 reads them
// coalesced along x and writes the uint8 result.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void resize_aa_h_kernel(const uint8_t* __restrict__ src, int layout, int T, int Hin, int Win,
                                                          int Wout, const int32_t* __restrict__ xmin, const int32_t* __restrict__ xsize,
                                                          const float* __restrict__ wx, int kx, float* __restrict__ tmp) {
  // one thread = one output column of one source row, all three colour channels: the taps are loaded once for the three
  // channels, and the tap table is TAP-MAJOR ([kx][Wout]) so that the lanes of a wave (consecutive xo) read consecutive floats
  const size_t total = (size_t)T * Hin * Wout;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int xo = (int)(i % Wout);
  const size_t r = i / Wout;
  const int y = (int)(r % Hin);
  const int t = (int)(r / Hin);
  const int x0 = xmin[xo], n = xsize[xo];
  const float* w = wx + xo;
  const size_t plane = (size_t)Hin * Wout;
  float* o = tmp + ((size_t)t * 3 * Hin + y) * Wout + xo;                                          // [T][3][Hin][Wout]
  if (layout == 0) {                                                                                // THWC: 3 adjacent bytes per pixel
    const uint8_t* p = src + (((size_t)t * Hin + y) * Win + x0) * 3;
    const float w0 = w[0];
    float a0 = __fmul_rn((float)p[0], w0), a1 = __fmul_rn((float)p[1], w0), a2 = __fmul_rn((float)p[2], w0);
    for (int j = 1; j < n; ++j) {
      const float wj = w[(size_t)j * Wout];
      a0 = fmaf((float)p[j * 3], wj, a0);
      a1 = fmaf((float)p[j * 3 + 1], wj, a1);
      a2 = fmaf((float)p[j * 3 + 2], wj, a2);
    }
    o[0] = a0; o[plane] = a1; o[2 * plane] = a2;
  } else {                                                                                          // TCHW
    const uint8_t* p = src + ((size_t)t * 3 * Hin + y) * Win + x0;
    const size_t cp = (size_t)Hin * Win;
    const float w0 = w[0];
    float a0 = __fmul_rn((float)p[0], w0), a1 = __fmul_rn((float)p[cp], w0), a2 = __fmul_rn((float)p[2 * cp], w0);
    for (int j = 1; j < n; ++j) {
      const float wj = w[(size_t)j * Wout];
      a0 = fmaf((float)p[j], wj, a0);
      a1 = fmaf((float)p[cp + j], wj, a1);
      a2 = fmaf((float)p[2 * cp + j], wj, a2);
    }
    o[0] = a0; o[plane] = a1; o[2 * plane] = a2;
  }
}

__global__ __launch_bounds__(256) void resize_aa_v_kernel(const float* __restrict__ tmp, int T, int Hin, int Hout, int Wout,
                                                          const int32_t* __restrict__ ymin, const int32_t* __restrict__ ysize,
                                                          const float* __restrict__ wy, int ky, uint8_t* __restrict__ dst) {
  const size_t total = (size_t)T * 3 * Hout * Wout;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int xo = (int)(i % Wout);
  size_t r = i / Wout;
  const int yo = (int)(r % Hout);
  const size_t tc = r / Hout;
  const int y0 = ymin[yo], n = ysize[yo];
  const float* w = wy + (size_t)yo * ky;
  const float* p = tmp + (tc * Hin + y0) * Wout + xo;
  float acc = __fmul_rn(p[0], w[0]);
  for (int j = 1; j < n; ++j) acc = fmaf(p[(size_t)j * Wout], w[j], acc);
  acc = fminf(fmaxf(acc, 0.f), 255.f);          // torchvision clamps the bicubic overshoot, then rounds half to even
  dst[i] = (uint8_t)rintf(acc);                 // [T][3][Hout][Wout]
}

// Both passes in one launch over output tiles of 64 columns x TH rows x 3 channels: the source window of a tile is staged in LDS by aligned
// dwords, the width pass leaves its fp32 rows in LDS, the height pass reads them there.  Same products in the same order as the two kernels
// above, so the same bytes.  Bound by vector instructions and the latency of a tile's three stages, not by bytes (a 720p pair is 5.5 MB in,
// 1.7 MB out).  The two launches spent 18.9 us on byte-wise global loads of the width pass (27 per output column) and 14.4 us on the height
// pass over an fp32 tensor of 12.6 MB that nothing else reads.  Here a lane owns a column and keeps its K weights (zero behind its own count)
// in registers for all rows of the tile, its 3 K source bytes are K dword reads shifted into place, and the height pass takes four columns a
// lane.  Two 720p frames to 392 x 728: 33.3 -> 11.6 us (rows x channels one column a lane: 15.9); two of 300 x 500: 15 -> 9.6; 24 of
// 1080p to 280 x 504 (17 taps, half of a tile's rows are its neighbour's too): 391 -> 138.  With the window from scalar loads, so that the source
// is asked for at once and not behind the tables' round trip and six reductions, and the tile's rows chosen for the launch (resize_plan), 16 or 8
// rows before: in a row of launches 10.5 -> 9.6, 8.8 -> 7.7 and 124 -> 112 us; 64 frames of 360p to 280 x 504: 83 -> 56; planar 480p pair: 10.2 -> 8.0.
// The tables are the caller's: a tile whose window does not fit what the host sized from the scale is computed tap by tap (same values).
constexpr int RS_COLS = 64;
constexpr int RS_WAVES = 8;
constexpr int RS_ROWS = 32;                     // output rows of a tile at most
constexpr int RS_LDS_MAX = 80 * 1024;          // two blocks on a compute unit
template <int K, bool PLANAR>
__global__ __launch_bounds__(RS_WAVES * 64) void resize_aa_tile_kernel(const uint8_t* __restrict__ src, int T, int Hin, int Win, uint8_t* __restrict__ dst,
                                                             int Hout, int Wout, const int32_t* __restrict__ xmin,
                                                             const int32_t* __restrict__ xsize, const float* __restrict__ wx,
                                                             const int32_t* __restrict__ ymin, const int32_t* __restrict__ ysize,
                                                             const float* __restrict__ wy, int ky, int TH, int rows_cap, int seg_dw) {
  constexpr int PX = PLANAR ? 1 : 3, NSEG = PLANAR ? 3 : 1;       // bytes from a pixel to the next; staged pieces of a source row
  extern __shared__ __attribute__((aligned(16))) float wrow[];    // [TH][ky up to 4s], then mid [rows_cap][3][64], then the pieces [rows_cap * NSEG][seg_dw]
  __shared__ int tap0[RS_ROWS], taps[RS_ROWS];
  float* mid = wrow + TH * ((ky + 3) & ~3);
  unsigned* raw = reinterpret_cast<unsigned*>(mid + (size_t)rows_cap * 3 * RS_COLS);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_x = (Wout + RS_COLS - 1) / RS_COLS, tiles_y = (Hout + TH - 1) / TH;
  const int tx = blockIdx.x % tiles_x, ty = (blockIdx.x / tiles_x) % tiles_y, t = blockIdx.x / (tiles_x * tiles_y);
  const int y0t = ty * TH, nrow = min(TH, Hout - y0t);
  const int xo = min(tx * RS_COLS + lane, Wout - 1), yl = y0t + min(lane, nrow - 1);
  // The window is that of the tile's first and last column and row (scalar loads: the staging below does not wait for the tables); a table in
  // which another one reaches beyond them takes the tap-by-tap form, as one whose window does not fit.
  typedef const __attribute__((address_space(4))) int* sptr;
  const sptr sx = (sptr)(uintptr_t)xmin, sy = (sptr)(uintptr_t)ymin, sn = (sptr)(uintptr_t)ysize;
  const int y_last = y0t + nrow - 1;
  const int lo = sx[tx * RS_COLS], hi = sx[min(tx * RS_COLS + RS_COLS, Wout) - 1], rlo = sy[y0t], rhi = sy[y_last] + max(sn[y_last], 1);
  const int x0 = xmin[xo], n = xsize[xo], yy = ymin[yl], yn = ysize[yl];
  const bool out = x0 < lo || x0 > hi || n > K || yy < rlo || yy + max(yn, 1) > rhi || yn > ky || yn < 1;          // every wave asks for all rows and columns
  const int cols = hi - lo + K, rows = rhi - rlo;
  const uint8_t* frame = src + (size_t)t * 3 * Hin * Win;
  const size_t plane = (size_t)Hin * Win;
  const bool live = tx * RS_COLS + lane < Wout;
  auto tap_by_tap = [&] {
    for (int it = wave; it < nrow * 3; it += RS_WAVES) {
      const int yo = y0t + it / 3, c = it - it / 3 * 3, ys = ymin[yo], ny = ysize[yo];
      float acc = 0.f;
      for (int i = 0; i < max(ny, 1); ++i) {
        const uint8_t* p = PLANAR ? frame + c * plane + (size_t)(ys + i) * Win + x0 : frame + ((size_t)(ys + i) * Win + x0) * 3 + c;
        float h = __fmul_rn((float)p[0], wx[xo]);
        for (int j = 1; j < n; ++j) h = fmaf((float)p[j * PX], wx[(size_t)j * Wout + xo], h);
        const float w = wy[(size_t)yo * ky + i];
        acc = i == 0 ? __fmul_rn(h, w) : fmaf(h, w, acc);
      }
      if (live) dst[(((size_t)t * 3 + c) * Hout + yo) * Wout + xo] = (uint8_t)rintf(fminf(fmaxf(acc, 0.f), 255.f));
    }
  };
  // block-uniform, and before anything is read through the tables: the window is inside the picture and what the host sized
  if (rows < 1 || rows > rows_cap || hi < lo || cols * PX + 8 > seg_dw * 4 || lo < 0 || lo >= Win || rlo < 0 || rhi > Hin) return tap_by_tap();
  float w[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const float f = wx[(size_t)j * Wout + xo];
    w[j] = (j == 0 || j < n) ? f : 0.f;                   // a tap behind the count adds 0 x byte: exact
  }
  // source window -> LDS.  A piece starts at the dword that holds its first byte and ends with the one that holds its last: every dword read
  // shares its word with a byte of the picture.
  const int nbytes = (min(lo + cols, Win) - lo) * PX, nseg = rows * NSEG;
  auto piece = [&](int sg) { return PLANAR ? frame + (sg % 3) * plane + (size_t)(rlo + sg / 3) * Win + lo : frame + ((size_t)(rlo + sg) * Win + lo) * 3; };
  for (int d0 = 0; d0 < seg_dw; d0 += 128)
    for (int s0 = wave; s0 < nseg; s0 += 8 * RS_WAVES) {
      unsigned v[8][2];
#pragma unroll
      for (int q = 0; q < 8; ++q) {                       // sixteen loads in flight per wave, clamped instead of predicated: a 720p tile arrives
        const uint8_t* p = piece(min(s0 + RS_WAVES * q, nseg - 1));          // in one round trip
        const unsigned sh = (unsigned)((uintptr_t)p & 3);
        const unsigned* pw = reinterpret_cast<const unsigned*>(p - sh);
        const int last = ((int)sh + nbytes - 1) >> 2;
        v[q][0] = pw[min(d0 + lane, last)];
        v[q][1] = pw[min(d0 + lane + 64, last)];
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int sg = s0 + RS_WAVES * q;
        if (sg < nseg) {
          if (d0 + lane < seg_dw) raw[sg * seg_dw + d0 + lane] = v[q][0];
          if (d0 + lane + 64 < seg_dw) raw[sg * seg_dw + d0 + lane + 64] = v[q][1];
        }
      }
    }
  // the height pass's weights, and where each row's taps begin and how many they are
  const int kyp = (ky + 3) & ~3;
  for (int i = threadIdx.x; i < nrow * kyp; i += RS_WAVES * 64) {
    const int r = i / kyp, j = i - r * kyp;
    wrow[i] = j < max(ysize[y0t + r], 1) ? wy[(size_t)(y0t + r) * ky + j] : 0.f;
  }
  if (wave == 0 && lane < nrow) { tap0[lane] = yy - rlo; taps[lane] = max(yn, 1); }
#pragma unroll
  for (int j = 0; j < K; ++j) asm volatile("" ::"v"(w[j]));          // the weights arrive under the staging, not behind it
  if (__builtin_amdgcn_ballot_w64(out) != 0) return tap_by_tap();      // block-uniform: every wave compared the same values
  __syncthreads();
  for (int r = wave; r < rows; r += RS_WAVES) {
    float a[3];
    if constexpr (PLANAR) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int b = (int)((uintptr_t)piece(r * 3 + c) & 3) + (x0 - lo);
        const unsigned* p = raw + (r * 3 + c) * seg_dw + (b >> 2);
        constexpr int ND = (K + 3) / 4;
        unsigned d[ND + 1];
#pragma unroll
        for (int i = 0; i <= ND; ++i) d[i] = p[i];
#pragma unroll
        for (int i = 0; i < ND; ++i) d[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], b & 3);
        float f = __fmul_rn((float)(d[0] & 255u), w[0]);
#pragma unroll
        for (int j = 1; j < K; ++j) f = fmaf((float)((d[j >> 2] >> (8 * (j & 3))) & 255u), w[j], f);
        a[c] = f;
      }
    } else {
      const int b = (int)((uintptr_t)piece(r) & 3) + (x0 - lo) * 3;
      const unsigned* p = raw + r * seg_dw + (b >> 2);
      constexpr int ND = (3 * K + 3) / 4;
      unsigned d[ND + 1];
#pragma unroll
      for (int i = 0; i <= ND; ++i) d[i] = p[i];
#pragma unroll
      for (int i = 0; i < ND; ++i) d[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], b & 3);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float f = __fmul_rn((float)((d[0] >> (8 * c)) & 255u), w[0]);
#pragma unroll
        for (int j = 1; j < K; ++j) { const int e = 3 * j + c; f = fmaf((float)((d[e >> 2] >> (8 * (e & 3))) & 255u), w[j], f); }
        a[c] = f;
      }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) mid[(r * 3 + c) * RS_COLS + lane] = a[c];
  }
  __syncthreads();
  // four columns a lane, sixteen lanes a row and channel: one 16-byte read and four products per tap
  const bool words = ((Wout & 3) | (int)((uintptr_t)dst & 3)) == 0;
  for (int task = threadIdx.x; task < nrow * 48; task += RS_WAVES * 64) {
    const int it = task >> 4, r = it / 3, c = it - r * 3, col = (task & 15) * 4, ny = taps[r];
    const float* wr = wrow + r * kyp;
    const float* p = mid + (tap0[r] * 3 + c) * RS_COLS + col;
    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < ny; j0 += 4) {
      const f32x4 w4 = *reinterpret_cast<const f32x4*>(wr + j0);
      f32x4 m[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) m[j] = *reinterpret_cast<const f32x4*>(p + min(j0 + j, ny - 1) * 3 * RS_COLS);      // behind the count: 0 x the last tap
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(m[j][e], w4[j], acc[e]);
    }
    unsigned o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (unsigned)rintf(fminf(fmaxf(acc[e], 0.f), 255.f));      // the bicubic overshoot is clamped, then half to even
    uint8_t* q = dst + (((size_t)t * 3 + c) * Hout + y0t + r) * Wout + tx * RS_COLS + col;
    const int left = Wout - (tx * RS_COLS + col);
    if (words) {
      if (left > 0) *reinterpret_cast<unsigned*>(q) = o[0] | (o[1] << 8) | (o[2] << 16) | (o[3] << 24);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < left) q[e] = (uint8_t)o[e];
    }
  }
}

template <int K>
static void launch_resize_tile(const uint8_t* src, int layout, int T, int Hin, int Win, uint8_t* dst, int Hout, int Wout, const int32_t* xmin,
                               const int32_t* xsize, const float* wx, const int32_t* ymin, const int32_t* ysize, const float* wy, int ky, int TH,
                               int rows_cap, int seg_dw, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)((size_t)T * ((Hout + TH - 1) / TH) * ((Wout + RS_COLS - 1) / RS_COLS)));
  static DeviceOnce attr_set;   // per instantiation
  if (attr_set.first()) {
    (void)hipFuncSetAttribute((const void*)resize_aa_tile_kernel<K, false>, hipFuncAttributeMaxDynamicSharedMemorySize, RS_LDS_MAX);
    (void)hipFuncSetAttribute((const void*)resize_aa_tile_kernel<K, true>, hipFuncAttributeMaxDynamicSharedMemorySize, RS_LDS_MAX);
  }
  if (layout == 0)
    resize_aa_tile_kernel<K, false><<<grid, dim3(RS_WAVES * 64), lds, st>>>(src, T, Hin, Win, dst, Hout, Wout, xmin, xsize, wx, ymin, ysize, wy, ky, TH, rows_cap, seg_dw);
  else
    resize_aa_tile_kernel<K, true><<<grid, dim3(RS_WAVES * 64), lds, st>>>(src, T, Hin, Win, dst, Hout, Wout, xmin, xsize, wx, ymin, ysize, wy, ky, TH, rows_cap, seg_dw);
}

// one launch while a tile's window fits RS_LDS_MAX with at least 8 rows: scales up to about 4 (tap tables of 5 to 17 columns); wider filters
// take the two passes, whose work does not grow with the overlap of neighbouring tiles
struct ResizePlan { int TH = 0, rows_cap = 0, seg_dw = 0; size_t lds = 0; };      // TH 0: two passes
static ResizePlan resize_plan(int layout, int T, int Hin, int Win, int Hout, int Wout, int kx, int ky) {
  ResizePlan p;
  if ((kx & 1) == 0 || kx < 5 || kx > 17) return p;
  const double sx = (double)Win / Wout, sy = (double)Hin / Hout;
  const int seg_dw = (((int)(63 * sx) + 2 + kx) * (layout == 0 ? 3 : 1) + 8 + 3) / 4;
  // rows a compute unit walks: tiles dealt to it x source rows of a tile.  More rows a tile: fewer source rows twice; fewer: an even share for all units
  // (two 720p frames to 392 x 728: 600 tiles of 16 rows put three on some units, 504 of 19 two on each: 10.5 -> 9.6 us; 64 of 360p to 280 x 504: 83 -> 56).
  long best = 0;
  for (int TH = 8; TH <= RS_ROWS; ++TH) {
    const int rows_cap = (int)((TH - 1) * sy + 4 * std::max(sy, 1.0)) + 3;
    const size_t lds = ((size_t)rows_cap * (3 * RS_COLS + (layout == 0 ? 1 : 3) * seg_dw) + TH * ((ky + 3) & ~3)) * 4;
    if (lds > RS_LDS_MAX) break;
    const long tiles = (long)T * ((Hout + TH - 1) / TH) * ((Wout + RS_COLS - 1) / RS_COLS), per = (tiles + 255) / 256;
    // a unit holds 160 KB and four blocks of eight waves: what is beyond runs behind
    const long fit = std::max<long>(1, std::min<long>(4, (long)(163840 / (lds + 512))));
    const long cost = (per + fit - 1) / fit * 12 + per * rows_cap;      // a round's latency: as long as some 12 source rows
    if (p.TH == 0 || cost < best) { p.TH = TH; p.rows_cap = rows_cap; p.seg_dw = seg_dw; p.lds = lds; best = cost; }
  }
  return p;
}
size_t resize_tmp_floats(int layout, int T, int Hin, int Win, int Hout, int Wout, int kx, int ky) {
  if (T <= 0 || Hin <= 0 || Win <= 0 || Hout <= 0 || Wout <= 0 || kx <= 0 || ky <= 0 || resize_plan(layout, T, Hin, Win, Hout, Wout, kx, ky).TH > 0) return 0;
  return (size_t)T * 3 * Hin * Wout;
}
int resize_bicubic_aa_u8(const uint8_t* src, int layout, int T, int Hin, int Win, uint8_t* dst, int Hout, int Wout,
                         const int32_t* xmin, const int32_t* xsize, const float* wx, int kx, const int32_t* ymin,
                         const int32_t* ysize, const float* wy, int ky, float* tmp, hipStream_t st) {
  if (T <= 0 || Hin <= 0 || Win <= 0 || Hout <= 0 || Wout <= 0 || kx <= 0 || ky <= 0 || (layout != 0 && layout != 1)) return LCC_ERR_SHAPE;
  const ResizePlan p = resize_plan(layout, T, Hin, Win, Hout, Wout, kx, ky);
  if (p.TH > 0) {
#define LCC_RS(KX) case KX: launch_resize_tile<KX>(src, layout, T, Hin, Win, dst, Hout, Wout, xmin, xsize, wx, ymin, ysize, wy, ky, p.TH, p.rows_cap, p.seg_dw, p.lds, st); return 0
    switch (kx) { LCC_RS(5); LCC_RS(7); LCC_RS(9); LCC_RS(11); LCC_RS(13); LCC_RS(15); LCC_RS(17); }
#undef LCC_RS
  }
  const size_t n1 = (size_t)T * Hin * Wout, n2 = (size_t)T * 3 * Hout * Wout;
  resize_aa_h_kernel<<<dim3((unsigned)((n1 + 255) / 256)), dim3(256), 0, st>>>(src, layout, T, Hin, Win, Wout, xmin, xsize, wx, kx, tmp);
  resize_aa_v_kernel<<<dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st>>>(tmp, T, Hin, Hout, Wout, ymin, ysize, wy, ky, dst);
  return 0;
}

}  // namespace lcc
