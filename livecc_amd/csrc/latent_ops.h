// Device code shared by latent.hip and decode_v2.hip.
#pragma once
#include "common.h"
#include "kernels.h"

namespace lcc {

LCC_DEVICE float dyt_value(float x, float alpha, float w, float b) { return fmaf(tanhf(alpha * x), w, b); }

// One new row behind the fused input projection, by a block of NT threads: part = fp32 slabs [nsplit][rows][ldn] with the columns
//   [0, qp) query latent | [qp, qp + rp) cache latent (rp = 0: the layer reads another layer's cache) | then one gate value per head.
// Writes the normed query latent (bf16 [rows][qp]; QUERY false: its consumer norms it), the normed cache latent straight into the slot's
// arena, and the sigmoid gates (fp32).  The padding columns are exact zeros (zero weight rows), so the sums of squares run over the padded
// widths and divide by the real ones.  red: 2 * NT / 64 floats of LDS.
template <int NT, bool QUERY>
LCC_DEVICE void latent_row(const LatentInArgs& a, int row, float* red) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const size_t slab = (size_t)a.rows * a.ldn;
  const float* src = a.part + (size_t)row * a.ldn;
  auto at = [&](int c) {
    f32x4 v = *reinterpret_cast<const f32x4*>(src + c);
    for (int s = 1; s < a.nsplit; ++s) v += *reinterpret_cast<const f32x4*>(src + s * slab + c);
    return v;
  };
  auto sq4 = [](f32x4 v) { return (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]); };
  // Bound by trips to memory: the first piece of either part (two slabs of it), its norm weights, the gates and the cache address are asked for at once,
  // at clamped addresses instead of behind branches, and the pieces stay in registers across the sums: 32 rows of 768 + 512
  // channels in two slabs, a launch of a decode step, 4.5 -> 3.6 us
  const int slot = a.rp > 0 ? a.tok_stream[row] : 0, c0 = tid * 4, zc = a.qp + a.rp + max(min(tid, a.heads - 1), -1);
  const int cq = QUERY ? min(c0, a.qp - 4) : 0, ck = a.rp > 0 ? a.qp + min(c0, a.rp - 4) : 0;
  const size_t second = a.nsplit > 1 ? slab : 0;
  auto first = [&](int c) { return *reinterpret_cast<const f32x4*>(src + c); };
  auto next = [&](int c) { return *reinterpret_cast<const f32x4*>(src + second + c); };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 vq = QUERY ? first(cq) : zero, vk = first(ck);
  const f32x4 uq = QUERY ? next(cq) : zero, uk = next(ck);
  u32x2 nq = {0u, 0u}, nk = {0u, 0u};
  if (QUERY) nq = ld8(a.q_norm + cq);
  if (a.rp > 0) nk = ld8(a.kv_norm + ck - a.qp);
  float z = src[zc];
  const float z1 = src[second + zc];
  bf16_t* dst = nullptr;
  if (a.rp > 0) dst = a.kv_base[slot] + a.kv_off + (size_t)(a.tok_pos ? a.tok_pos[row] : a.kv_len[slot]) * a.rp;
  if (a.nsplit > 1) { vq += uq; vk += uk; z += z1; }
  for (int s = 2; s < a.nsplit; ++s) {
    if (QUERY) vq += *reinterpret_cast<const f32x4*>(src + s * slab + cq);
    vk += *reinterpret_cast<const f32x4*>(src + s * slab + ck);
    z += src[s * slab + zc];
  }
  if (!QUERY || c0 >= a.qp) vq = zero;
  if (c0 >= a.rp) vk = zero;
  float sq = sq4(vq), sk = sq4(vk);
  if (QUERY)
    for (int c = c0 + NT * 4; c < a.qp; c += NT * 4) sq += sq4(at(c));
  for (int c = c0 + NT * 4; c < a.rp; c += NT * 4) sk += sq4(at(a.qp + c));
  sq = wave_sum(sq); sk = wave_sum(sk);
  if (lane == 0) { red[wave] = sq; red[NW + wave] = sk; }
  for (int h = tid; h < a.heads; h += NT) {
    if (h != tid) {
      z = src[a.qp + a.rp + h];
      for (int s = 1; s < a.nsplit; ++s) z += src[s * slab + a.qp + a.rp + h];
    }
    a.gate[(size_t)row * a.heads + h] = 1.f / (1.f + expf(-z));
  }
  __syncthreads();
  sq = 0.f; sk = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) { sq += red[w]; sk += red[NW + w]; }
  auto put = [&](bf16_t* to, u32x2 w, int c, f32x4 v, float inv) {
    st8(to + c, (u32x2){pack2(v[0] * inv * lo2f(w.x), v[1] * inv * hi2f(w.x)), pack2(v[2] * inv * lo2f(w.y), v[3] * inv * hi2f(w.y))});
  };
  if (QUERY) {
    const float iq = 1.f / sqrtf(sq / (float)a.q_rank + a.eps);
    bf16_t* to = a.cq + (size_t)row * a.qp;
    if (c0 < a.qp) put(to, nq, c0, vq, iq);
    for (int c = c0 + NT * 4; c < a.qp; c += NT * 4) put(to, ld8(a.q_norm + c), c, at(c), iq);
  }
  const float ik = a.rp > 0 ? 1.f / sqrtf(sk / (float)a.kv_rank + a.eps) : 0.f;
  if (c0 < a.rp) put(dst, nk, c0, vk, ik);
  for (int c = c0 + NT * 4; c < a.rp; c += NT * 4) put(dst, ld8(a.kv_norm + c), c, at(a.qp + c), ik);
}

}  // namespace lcc
