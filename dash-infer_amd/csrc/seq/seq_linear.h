// seq_linear.h -- what the kernels of dihip_linear (seq_linear.hip, seq_linear_tile.hip) share: arguments and epilogue
#pragma once
#include "seq_common.h"

namespace dihip {

struct LinArgs {
  const void* x; long ldx, xg; int xgroups;
  const void* w; const void* bias;
  void* y; long ldy, yg;
  const float* mul; long ldm;
  int T, N, K, act, act_lo, act_hi, ydt, round_ops;
  int mul_group; float act_param;               // mul holds one number per group; the parameter of an activation that has one
  const int32_t* seg; const int32_t* row_map;   // segmented form: group g owns the output rows seg[g] .. seg[g + 1], row r reads x row row_map[r]
  const void* w2;                               // gated form: y = act(x . w^T) * (x . w2^T); w2 is shaped as w.  No groups, bias or mul
  // residual form (res): y is the f32 residual stream, y += res_a + result, and, with norm_w, h16 = bf16(tanh(norm_alpha * y) * norm_w + norm_b), rows of N.  No groups
  int res; const float* res_a; long res_lda; float norm_alpha; const void* norm_w; const void* norm_b; uint16_t* h16;   // (res_a NULL: the result alone; norm: bf16)
};

// the residual form's way out (the arithmetic of dihip_add_dyt, step by step)
struct LinRes { float x, a, w, b; };
__device__ __forceinline__ LinRes lin_res_load(const LinArgs& q, int t, int n) {
  LinRes r{((const float*)q.y)[(size_t)t * q.ldy + n], 0.f, 0.f, 0.f};
  if (q.res_a) r.a = q.res_a[(size_t)t * q.res_lda + n];
  if (q.norm_w) { r.w = bf16_bits_to_f32(((const uint16_t*)q.norm_w)[n]); r.b = bf16_bits_to_f32(((const uint16_t*)q.norm_b)[n]); }
  return r;
}
__device__ __forceinline__ void lin_res_store(const LinArgs& q, int t, int n, float v, const LinRes& r) {
  const float x = r.x + (q.res_a ? r.a + v : v);
  ((float*)q.y)[(size_t)t * q.ldy + n] = x;
  if (q.norm_w) q.h16[(size_t)t * q.N + n] = (uint16_t)f32_to_bf16_bits(tanhf(q.norm_alpha * x) * r.w + r.b);
}

// the rows of group g: [lo, hi)
__device__ __forceinline__ void lin_rows(const LinArgs& a, int g, int& lo, int& hi) {
  lo = 0; hi = a.T;
  if (a.seg) { lo = a.seg[g]; hi = a.seg[g + 1]; }
}
__device__ __forceinline__ size_t lin_xrow(const LinArgs& a, int r) { return (size_t)(a.row_map ? a.row_map[r] : r); }

// RES_TOO: a.res may be set.  (The residual form's code in an unrolled epilogue of 16 pieces -- linear_mfma_kernel -- kept the compiler from unrolling it: the sums went through scratch memory)
template <bool RES_TOO = true>
__device__ __forceinline__ void lin_epilogue(const LinArgs& a, int g, int t, int n, float v, int wdt) {
  if (a.bias) v += ld_any(a.bias, (size_t)g * a.N + n, wdt);
  const int col = g * a.N + n;
  if (col >= a.act_lo && col < a.act_hi) v = a.act == DIHIP_SEQ_ACT_SOFTCAP ? a.act_param * tanhf(v / a.act_param) : apply_act(v, a.act);
  const size_t o = (size_t)t * a.ldy + (size_t)g * a.yg + n;
  if (a.mul) v *= a.mul[(size_t)t * a.ldm + (a.mul_group ? (size_t)g : (size_t)g * a.yg + n)];
  if (RES_TOO && a.res) return lin_res_store(a, t, n, v, lin_res_load(a, t, n));
  st_any(a.y, o, a.ydt, v);
}

// the same for 4 neighbouring columns n .. n + 3 of row t; n is a multiple of 4.  vec4 (lin_vec4): N, strides and addresses allow 16-byte (f32) /
// 8-byte (bf16) pieces, else one column after the other.  bias: bf16
inline bool lin_vec4(const LinArgs& a) {
  const bool mul = !a.mul || a.mul_group || ((reinterpret_cast<uintptr_t>(a.mul) & 15) == 0 && a.ldm % 4 == 0);
  return a.N % 4 == 0 && a.ldy % 4 == 0 && a.yg % 4 == 0 && (reinterpret_cast<uintptr_t>(a.y) & (a.ydt == DIHIP_F32 ? 15 : 7)) == 0 && mul &&
         (!a.bias || (reinterpret_cast<uintptr_t>(a.bias) & 7) == 0) &&
         (!a.res || ((!a.res_a || ((reinterpret_cast<uintptr_t>(a.res_a) & 15) == 0 && a.res_lda % 4 == 0)) &&
                     ((reinterpret_cast<uintptr_t>(a.norm_w) | reinterpret_cast<uintptr_t>(a.norm_b) | reinterpret_cast<uintptr_t>(a.h16)) & 7) == 0));
}
__device__ __forceinline__ f32x4_t lin_bias4(const LinArgs& a, int g, int n, bool vec4) {
  if (!vec4 || !a.bias || n >= a.N) return f32x4_t{0.f, 0.f, 0.f, 0.f};
  const u32x2_t u = *reinterpret_cast<const u32x2_t*>((const uint16_t*)a.bias + (size_t)g * a.N + n);
  return f32x4_t{bf16_bits_to_f32(u[0] & 0xffffu), bf16_bits_to_f32(u[0] >> 16), bf16_bits_to_f32(u[1] & 0xffffu), bf16_bits_to_f32(u[1] >> 16)};
}
// the residual form's: columns n .. n + 3 of row t, the product's sums v and nothing else on them
__device__ __forceinline__ void lin_res4(const LinArgs& a, int t, int n, f32x4_t v, bool vec4) {
  if (!vec4) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < a.N) lin_res_store(a, t, n + r, v[r], lin_res_load(a, t, n + r));
    return;
  }
  if (n >= a.N) return;
  f32x4_t* y = reinterpret_cast<f32x4_t*>((float*)a.y + (size_t)t * a.ldy + n);
  f32x4_t x = *y;
  if (a.res_a) v = *reinterpret_cast<const f32x4_t*>(a.res_a + (size_t)t * a.res_lda + n) + v;
  x += v;
  *y = x;
  if (a.norm_w) {
    const u32x2_t w = *reinterpret_cast<const u32x2_t*>((const uint16_t*)a.norm_w + n), b2 = *reinterpret_cast<const u32x2_t*>((const uint16_t*)a.norm_b + n);
    uint32_t h[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      h[r] = f32_to_bf16_bits(tanhf(a.norm_alpha * x[r]) * bf16_bits_to_f32((w[r >> 1] >> (r & 1) * 16) & 0xffffu) + bf16_bits_to_f32((b2[r >> 1] >> (r & 1) * 16) & 0xffffu));
    *reinterpret_cast<u32x2_t*>(a.h16 + (size_t)t * a.N + n) = u32x2_t{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
  }
}
template <bool RES_TOO = true>
__device__ __forceinline__ void lin_epilogue4(const LinArgs& a, int g, int t, int n, f32x4_t v, const f32x4_t& bias, bool vec4) {
  if (RES_TOO && a.res) return lin_res4(a, t, n, v, vec4);   // (uniform; no bias, activation or factor beside it)
  if (!vec4) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < a.N) lin_epilogue<false>(a, g, t, n + r, v[r], DIHIP_BF16);
    return;
  }
  if (n >= a.N) return;
  if (a.bias) v += bias;
  const int col = g * a.N + n;
  if (col + 3 >= a.act_lo && col < a.act_hi) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (col + r >= a.act_lo && col + r < a.act_hi) v[r] = a.act == DIHIP_SEQ_ACT_SOFTCAP ? a.act_param * tanhf(v[r] / a.act_param) : apply_act(v[r], a.act);
  }
  if (a.mul) {
    if (a.mul_group) v *= a.mul[(size_t)t * a.ldm + g];
    else v *= *reinterpret_cast<const f32x4_t*>(a.mul + (size_t)t * a.ldm + (size_t)g * a.yg + n);
  }
  const size_t o = (size_t)t * a.ldy + (size_t)g * a.yg + n;
  if (a.ydt == DIHIP_F32) *reinterpret_cast<f32x4_t*>((float*)a.y + o) = v;
  else *reinterpret_cast<u32x2_t*>((uint16_t*)a.y + o) = u32x2_t{f32_to_bf16_bits(v[0]) | (f32_to_bf16_bits(v[1]) << 16),
                                                                  f32_to_bf16_bits(v[2]) | (f32_to_bf16_bits(v[3]) << 16)};
}

// the gated form's: g and u are the sums of columns n .. n + 3 with w and with w2
__device__ __forceinline__ void lin_gated4(const LinArgs& a, int t, int n, f32x4_t g, const f32x4_t& u, bool vec4) {
  if (n >= a.N) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) g[r] = apply_act(g[r], a.act) * u[r];
  const size_t o = (size_t)t * a.ldy + n;
  if (!vec4) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < a.N) st_any(a.y, o + r, a.ydt, g[r]);
  } else if (a.ydt == DIHIP_F32) {
    *reinterpret_cast<f32x4_t*>((float*)a.y + o) = g;
  } else {
    *reinterpret_cast<u32x2_t*>((uint16_t*)a.y + o) = u32x2_t{f32_to_bf16_bits(g[0]) | (f32_to_bf16_bits(g[1]) << 16),
                                                              f32_to_bf16_bits(g[2]) | (f32_to_bf16_bits(g[3]) << 16)};
  }
}

__device__ __forceinline__ f32x4_t mfma_bf16(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// seq_linear_tile.hip: bf16 rows times bf16 weights in pipelined tiles.  ok: the shape is taken (K % 64 == 0; the caller checks types and 16-byte
// alignment); slab: bytes of workspace for the K parts (0: not split)
struct LinTilePlan {
  bool ok;
  int shape;           // of the tiles (seq_linear_tile.hip)
  int parts;
  size_t slab;
};
// the slab of one K part: [row][group][column], every row of a group padded to whole 4 columns (the gated form: its two matrices as two groups)
inline size_t lin_slab_part_bytes(int T, int N, int groups) { return (size_t)T * groups * (((size_t)N + 3) & ~(size_t)3) * sizeof(float); }
LinTilePlan plan_linear_tile(int Tg, int N, int K, int groups, long ldx, bool split, bool gated = false);   // (gated: N columns of each matrix, groups 1)
int launch_linear_tile(const LinArgs& a, const LinTilePlan& p, int Tg, int groups, float* slab, hipStream_t s);

}  // namespace dihip
