// seq_linear.hip -- dihip_linear: y = epilogue(x . W^T + bias) for row-major [N, K] weights as checkpoints store them,
// grouped (block-diagonal / per-head) forms included.  The kernels:
//   linear_tile_kernel   every product and sum in f32, k ascending (DIHIP_MATH_F32; also any operand type / odd shape)
//   linear_pipe_kernel   bf16 operands on the matrix cores, pipelined tiles of eleven sizes, K split where tiles are few (seq_linear_tile.hip)
//   linear_mfma_kernel   the same for f32 rows (rounded to bf16), K % 64 != 0 or unaligned operands: 128 x 128 x 32 tiles through registers (segments of a few
//                        tokens too where that is faster: seg_in_tiles)
//   linear_stream_lds_kernel  bf16 operands, 2 .. 64 rows, K % 64 == 0 and 1024 or more (segments: 512): both streamed through LDS, K split over a workgroup's waves
//   linear_stream_kernel the same for f32 rows and other K: weights straight from memory into the matrix cores
//   linear_row_kernel    one row (decode), bf16 operands: two workgroups per CU walk the weight rows past x in registers
//   linear_skinny_kernel one short row, one row per group, a few rows where that is faster (skinny_rows) or the products are f32: a streamed weight, one wave
//                        per 2 weight rows, 4 rows at a time
//   linear_fewcols_kernel a router's logits
// dihip_linear_gated (act(x . w^T) * (x . w2^T)) runs in forms of linear_pipe, linear_stream_lds and linear_row_kernel that walk both matrices in one launch.
// f32 products: an output element is one chain over k, ascending, whatever T is.  bf16 products: the order of its f32 sum follows the kernel, which T chooses (one
// row; 2 .. 64; more), and in linear_pipe_kernel the number of K parts, which T chooses too: results of other row counts are equal within f32 rounding,
// not to the bit.  Within 2 .. 64 rows of one kernel, and above 64 where K is in one part (segments: always), T does not matter.
#include <algorithm>
#include <type_traits>
#include "seq_linear.h"

namespace dihip {
namespace {

// ------------------------------------------------------------------------------------------ exact f32 tile kernel
template <int XT, int WT>
__global__ __launch_bounds__(256) void linear_tile_kernel(LinArgs a) {
  __shared__ float xs[16][68];
  __shared__ float ws[16][68];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int g = blockIdx.z, n0 = blockIdx.x * 64;
  int t_lo, t_hi;
  lin_rows(a, g, t_lo, t_hi);
  const int m0 = t_lo + blockIdx.y * 64;
  if (m0 >= t_hi) return;
  const size_t xoff = (size_t)(g % a.xgroups) * a.xg;
  const size_t wbase = (size_t)g * a.N * a.K;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < a.K; k0 += 16) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int idx = tid + 256 * j, r = idx >> 4, kk = idx & 15;
      float xv = 0.f, wv = 0.f;
      if (k0 + kk < a.K) {
        if (m0 + r < t_hi) xv = load_ft<XT>(a.x, lin_xrow(a, m0 + r) * a.ldx + xoff + k0 + kk);
        if (n0 + r < a.N) wv = load_ft<WT>(a.w, wbase + (size_t)(n0 + r) * a.K + k0 + kk);
      }
      if (a.round_ops) { xv = ft_round<DIHIP_BF16>(xv); wv = ft_round<DIHIP_BF16>(wv); }
      xs[kk][r] = xv;
      ws[kk][r] = wv;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const f32x4_t av = *reinterpret_cast<const f32x4_t*>(&xs[kk][ty * 4]);
      const f32x4_t bv = *reinterpret_cast<const f32x4_t*>(&ws[kk][tx * 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(av[i], bv[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = m0 + ty * 4 + i;
    if (t >= t_hi) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < a.N) lin_epilogue<false>(a, g, t, n, acc[i][j], WT);
    }
  }
}

// ------------------------------------------------------------------------------------------ bf16 matrix-core kernel
// 8 consecutive k of one row as packed bf16; VEC: the 8 are in range and 16-byte aligned (host-checked), else guarded
template <int XT, bool VEC>
__device__ __forceinline__ u32x4_t load8_bf16(const void* p, size_t i, int kleft, bool row_ok) {
  u32x4_t r = {0u, 0u, 0u, 0u};
  if (!row_ok || kleft <= 0) return r;
  if constexpr (VEC) {
    if constexpr (XT == DIHIP_F32) {
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>((const float*)p + i);
      const f32x4_t hi = *reinterpret_cast<const f32x4_t*>((const float*)p + i + 4);
      r[0] = pack_bf16x2(lo[0], lo[1]); r[1] = pack_bf16x2(lo[2], lo[3]);
      r[2] = pack_bf16x2(hi[0], hi[1]); r[3] = pack_bf16x2(hi[2], hi[3]);
    } else {
      r = *reinterpret_cast<const u32x4_t*>((const uint16_t*)p + i);
    }
  } else {
    uint32_t e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = j < kleft ? f32_to_bf16_bits(load_ft<XT>(p, i + j)) : 0u;
    r[0] = e[0] | (e[1] << 16); r[1] = e[2] | (e[3] << 16); r[2] = e[4] | (e[5] << 16); r[3] = e[6] | (e[7] << 16);
  }
  return r;
}

// RES: the residual form, a kernel of its own: its code beside the other epilogue's was too much to unroll, the sums were indexed in scratch memory (f32 rows, 2048 of 4096 ->
// 4096 188 -> 687 us)
template <int XT, bool VEC, bool RES>
__global__ __launch_bounds__(256) void linear_mfma_kernel(LinArgs a, bool vec4) {
  constexpr int BK = 32, UPR = BK / 8, UN = 128 * UPR / 256;   // k per step (64 measured slower: fewer workgroups per CU), 16-byte units per tile row, units per thread
  constexpr int LD = BK + 8;  // bf16 elements per LDS row: 8 of padding (80 bytes: 16-byte aligned fragments)
  __shared__ __attribute__((aligned(16))) uint16_t As[128 * LD];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[128 * LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int g = blockIdx.z, n0 = blockIdx.x * 128;
  int t_lo, t_hi;
  lin_rows(a, g, t_lo, t_hi);
  const int m0 = t_lo + blockIdx.y * 128;
  if (m0 >= t_hi) return;
  const size_t xoff = (size_t)(g % a.xgroups) * a.xg;
  const size_t wbase = (size_t)g * a.N * a.K;
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = z4;
  u32x4_t ra[UN], rb[UN];
  size_t xrow[UN];   // the x row of each of the thread's units: fixed for the whole walk
#pragma unroll
  for (int j = 0; j < UN; ++j) {
    const int r = (tid + 256 * j) / UPR;
    xrow[j] = m0 + r < t_hi ? lin_xrow(a, m0 + r) : 0;
  }
  auto fetch = [&](int k0) {
#pragma unroll
    for (int j = 0; j < UN; ++j) {
      const int u = tid + 256 * j, r = u / UPR, k = k0 + (u % UPR) * 8;
      ra[j] = load8_bf16<XT, VEC>(a.x, xrow[j] * a.ldx + xoff + k, a.K - k, m0 + r < t_hi);
      rb[j] = load8_bf16<DIHIP_BF16, VEC>(a.w, wbase + (size_t)(n0 + r) * a.K + k, a.K - k, n0 + r < a.N);
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < a.K; k0 += BK) {
#pragma unroll
    for (int j = 0; j < UN; ++j) {
      const int u = tid + 256 * j, r = u / UPR, kq = (u % UPR) * 8;
      *reinterpret_cast<u32x4_t*>(&As[r * LD + kq]) = ra[j];
      *reinterpret_cast<u32x4_t*>(&Bs[r * LD + kq]) = rb[j];
    }
    __syncthreads();
    if (k0 + BK < a.K) fetch(k0 + BK);
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      u32x4_t af[4], bf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        af[i] = *reinterpret_cast<const u32x4_t*>(&As[(wm * 64 + i * 16 + (lane & 15)) * LD + ks * 32 + (lane >> 4) * 8]);
        bf[i] = *reinterpret_cast<const u32x4_t*>(&Bs[(wn * 64 + i * 16 + (lane & 15)) * LD + ks * 32 + (lane >> 4) * 8]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma_bf16(bf[j], af[i], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {   // a lane holds 4 neighbouring columns
    const int n = n0 + wn * 64 + j * 16 + (lane >> 4) * 4;
    const f32x4_t b = lin_bias4(a, g, n, vec4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = m0 + wm * 64 + i * 16 + (lane & 15);
      if (t >= t_hi) continue;
      if constexpr (RES) lin_res4(a, t, n, acc[i][j], vec4);
      else lin_epilogue4<false>(a, g, t, n, acc[i][j], b, vec4);
    }
  }
}

// ------------------------------------------------------------------------------------------ weight-streaming kernel, matrix cores
// Up to 64 rows against weights that are read once (decoding steps of a batch, short portions).  Bound by the weights' bytes and by what the
// workgroups pull of the activations, so everything serves the loads in flight:
//   * a workgroup owns ROWS weight rows and its WV waves split K among them (block b of 128 elements belongs to wave b % WV): a narrow
//     matrix still gives every wave a stream of its own, and at any time the workgroup reads adjacent blocks of the same rows;
//   * weights and activations go straight from memory into MFMA operands (the weight rows are the A operand: a lane ends with 4
//     neighbouring columns of one output row); a wave issues all loads of a block before the first product, and with PRE the weights of
//     its next block as well.  Nothing is staged, no barrier before the end: the activations (T x K bf16) live in the L2s;
//   * the waves' partial sums meet in LDS and are added in the order of the waves: an element's sum does not depend on the rows beside it.
// 24 rows: 8192 -> 2048 180 -> 23 us, 2048 -> 8192 57 -> 13, 4096 -> 14336 100 -> 39, 4096 -> 32000 104 -> 70 (before: 128 x 128 tiles).  What is left is the activations:
// each workgroup pulls T x K of them from its L2 for ROWS x K weights.
// K % 8 == 0 and 16-byte aligned rows (host-checked).
template <int XT>
__device__ __forceinline__ u32x4_t stream_x(const char* p, bool ok) {
  u32x4_t r = {0u, 0u, 0u, 0u};
  if (ok) {
    if constexpr (XT == DIHIP_F32) {
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(p), hi = *reinterpret_cast<const f32x4_t*>(p + 16);
      r = u32x4_t{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]), pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
    } else {
      r = *reinterpret_cast<const u32x4_t*>(p);
    }
  }
  return r;
}

constexpr int STREAM_MAX_ROWS = 64;
constexpr int STREAM_SPLIT_K = 256;   // shorter walks are not split

template <int XT, int ROWS, int TF, int WV, bool PRE>
__global__ __launch_bounds__(64 * WV, (ROWS * TF > 64 || XT == DIHIP_F32) ? 2 : 4) void linear_stream_kernel(LinArgs a, bool vec4) {
  constexpr int RF = ROWS / 16, U = 4, BK = U * 32;
  constexpr int XE = XT == DIHIP_F32 ? 4 : 2;
  __shared__ __attribute__((aligned(16))) f32x4_t red[WV][RF * TF][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i16 = lane & 15, q = lane >> 4;
  const int g = blockIdx.y, n0 = blockIdx.x * ROWS;
  int lo, hi;
  lin_rows(a, g, lo, hi);
  if (lo >= hi) return;
  const int count = min(hi - lo, 16 * TF);
  const uint16_t* wp[RF];   // rows past N re-read the last one, rows past the group's the last of those: never stored
#pragma unroll
  for (int r = 0; r < RF; ++r) wp[r] = (const uint16_t*)a.w + ((size_t)g * a.N + min(n0 + r * 16 + i16, a.N - 1)) * a.K + q * 8;
  const char* xp[TF];
#pragma unroll
  for (int t = 0; t < TF; ++t)
    xp[t] = (const char*)a.x + (lin_xrow(a, lo + min(t * 16 + i16, count - 1)) * a.ldx + (size_t)(g % a.xgroups) * a.xg + q * 8) * XE;
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[RF][TF];
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int t = 0; t < TF; ++t) acc[r][t] = z4;
  auto walk = [&](auto whole) {   // WHOLE: K is a multiple of the block; else lanes past K read nothing and multiply zeros
    constexpr bool WHOLE = decltype(whole)::value;
    auto load_w = [&](u32x4_t (&w)[U][RF], int k) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < RF; ++r) {
          if constexpr (!WHOLE) w[u][r] = u32x4_t{0u, 0u, 0u, 0u};
          if (WHOLE || k + u * 32 + q * 8 < a.K) w[u][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wp[r] + k + u * 32));
        }
    };
    u32x4_t w[U][RF], wn[U][RF];
    // a short K is one wave's: the sum of the tile kernel, bit for bit
    const int first = a.K >= STREAM_SPLIT_K ? wave * BK : (wave == 0 ? 0 : a.K), step = a.K >= STREAM_SPLIT_K ? WV * BK : BK;
    if (PRE && first < a.K) load_w(w, first);
    for (int k = first; k < a.K; k += step) {
      u32x4_t x[U][TF];
      if constexpr (!PRE) load_w(w, k);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < TF; ++t) x[u][t] = stream_x<XT>(xp[t] + (size_t)(k + u * 32) * XE, WHOLE || k + u * 32 + q * 8 < a.K);
      if (PRE && k + step < a.K) load_w(wn, k + step);   // (uniform)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < RF; ++r) {
#pragma unroll
          for (int t = 0; t < TF; ++t) acc[r][t] = mfma_bf16(w[u][r], x[u][t], acc[r][t]);
          if constexpr (PRE) w[u][r] = wn[u][r];
        }
    }
  };
  if (a.K % BK == 0) walk(std::true_type{});
  else walk(std::false_type{});
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int t = 0; t < TF; ++t) red[wave][r * TF + t][lane] = acc[r][t];
  __syncthreads();
  for (int e = tid; e < RF * TF * 64; e += 64 * WV) {   // 4 neighbouring columns of one row
    const int f = e >> 6, l = e & 63, t = (f % TF) * 16 + (l & 15), n = n0 + (f / TF) * 16 + (l >> 4) * 4;
    if (t >= count) continue;
    f32x4_t v = red[0][f][l];
#pragma unroll
    for (int i = 1; i < WV; ++i) v += red[i][f][l];
    lin_epilogue4(a, g, lo + t, n, v, lin_bias4(a, g, n, vec4), vec4);
  }
}

// The same walk for bf16 rows with K % 64 == 0, by LDS: what binds the form above is the number of pieces that its loads touch (an operand is 16 rows x
// 64 bytes), not the bytes.  Here a wave brings its blocks of 64 elements -- pieces of 8 rows x 128 bytes, whole cache lines -- straight into LDS of its own (D blocks
// deep, no barrier: only the wave itself waits for its loads) and reads the operands from there.  Piece and swizzle as in linear_pipe_kernel.
// 24 rows, the form above -> this, us: 8192 -> 2048 23.0 -> 15.4, 2048 -> 8192 13.4 -> 10.6, 4096 -> 14336 38.6 -> 25.7, 4096 -> 32000 69.6 -> 58; 64 rows 45.7 -> 22.2,
// 17.8 -> 13.1, 56.3 -> 29.9, 90 -> 63.  (The form above with its blocks asked for one ahead of the other was slower: it does not wait for latency.)
// SEG: segments of rows, which a map may name: they may lie anywhere, 64-bit addresses per lane; and as many row operands as the segment needs, often far fewer
// than the bound that TF was chosen for (copies of its last row would be half of what is brought).  Gathered [gate | up] products of 64 experts, 6 per token, 2048 -> 2816, the form
// above -> this: 2 / 8 / 17 / 64 tokens 32.4 / 87 / 164 / 193 -> 26.2 / 79 / 114 / 139.
constexpr int STREAM_LDS_WAVES = 4;
// GATED (linear_gated): the first half of the workgroup's weight rows are w's, the second the same ones of w2.
template <int ROWS, int TF, int WV, int D, bool SEG, bool GATED>
__global__ __launch_bounds__(64 * WV, 2) void linear_stream_lds_kernel(LinArgs a, bool vec4) {
  constexpr int RF = (ROWS + 15) / 16, WP = ROWS / 8, PER = WP + 2 * TF, SLOT = PER * 1024, COLS = GATED ? ROWS / 2 : ROWS;   // (WP: pieces of weights; COLS: of y)
  static_assert(ROWS >= 16 || !GATED, "both halves are whole pieces");
  static_assert((D - 1) * PER < 64, "what is in flight is counted");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.y, n0 = blockIdx.x * COLS;
  int lo, hi;
  lin_rows(a, g, lo, hi);
  if (lo >= hi) return;
  const int count = min(hi - lo, 16 * TF);
  const int prow = lane >> 3, pchunk = (lane & 7) ^ prow;
  const char* wbase = (const char*)((const uint16_t*)a.w + ((size_t)g * a.N + n0) * a.K);
  const char* w2base = GATED ? (const char*)((const uint16_t*)a.w2 + (size_t)n0 * a.K) : nullptr;
  const char* xbase = (const char*)((const uint16_t*)a.x + (size_t)(g % a.xgroups) * a.xg);
  uint32_t off[PER];   // (the host checks that they fit); rows past N re-read the last one, rows past the group's the last of those: never stored
  const char* xaddr[2 * TF];   // (SEG: of the next block)
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int r = (p < WP ? p : p - WP) * 8 + prow;
    if (p < WP) {
      off[p] = (uint32_t)min(r % COLS, a.N - 1 - n0) * (uint32_t)a.K * 2 + pchunk * 16;
    } else {
      const size_t from = lin_xrow(a, lo + min(r, count - 1)) * a.ldx * 2 + pchunk * 16;
      if constexpr (SEG) xaddr[p - WP] = xbase + from + wave * 128;
      else off[p] = (uint32_t)from;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + wave * D * SLOT;
  const unsigned char* mine = lds + wave * D * SLOT;
  const int blocks = a.K / 64, steps = (blocks - wave + WV - 1) / WV;   // blocks wave, wave + WV, ..
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[RF][TF];
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int t = 0; t < TF; ++t) acc[r][t] = z4;
  const int f0 = (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) * 16);
  const int fw = ROWS == 8 ? f0 & ~1024 : f0;   // (8 weight rows: twice in their operand)
  auto ring = [&](auto used) {   // with the first TN row operands
    constexpr int TN = decltype(used)::value, USED = WP + 2 * TN;
    auto fetch = [&](int i, int slot) {   // (called for i = 0, 1, 2, ..)
      const char* wk = wbase + (size_t)(wave + i * WV) * 128;
      const char* w2k = GATED ? w2base + (size_t)(wave + i * WV) * 128 : wk;
      const char* xk = xbase + (size_t)(wave + i * WV) * 128;
#pragma unroll
      for (int p = 0; p < USED; ++p) {
        const uint32_t to = lds0 + slot * SLOT + p * 1024;
        if (SEG && p >= WP) {
          const char* const from = xaddr[p - WP];
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(from) : "memory");
          xaddr[p - WP] += WV * 128;
        } else {
          const uint32_t o = off[p];
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(o), "s"(p < (GATED ? WP / 2 : WP) ? wk : p < WP ? w2k : xk) : "memory");
        }
      }
    };
    auto mul = [&](int slot) {
      const unsigned char* b = mine + slot * SLOT;
      u32x4_t w[2][RF], x[2][TN];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int r = 0; r < RF; ++r) w[h][r] = *reinterpret_cast<const u32x4_t*>(b + r * 2048 + (h ? fw ^ 64 : fw));
#pragma unroll
        for (int t = 0; t < TN; ++t) x[h][t] = *reinterpret_cast<const u32x4_t*>(b + WP * 1024 + t * 2048 + (h ? f0 ^ 64 : f0));
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < RF; ++r)
#pragma unroll
          for (int t = 0; t < TN; ++t) acc[r][t] = mfma_bf16(w[h][r], x[h][t], acc[r][t]);
    };
    if (steps >= D) {
#pragma unroll
      for (int i = 0; i < D; ++i) fetch(i, i);
      int slot = 0;
      for (int i = 0; i + D < steps; ++i) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * USED) : "memory");
        mul(slot);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot has been read
        fetch(i + D, slot);
        slot = slot + 1 == D ? 0 : slot + 1;
      }
#pragma unroll
      for (int j = 0; j < D; ++j) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1 - j) * USED) : "memory");
        mul(slot);
        slot = slot + 1 == D ? 0 : slot + 1;
      }
    } else {
      for (int i = 0; i < steps; ++i) fetch(i, i);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      for (int i = 0; i < steps; ++i) mul(i);
    }
  };
  if (SEG && TF > 1 && count <= 16) ring(std::integral_constant<int, 1>{});
  else if (SEG && TF > 2 && count <= 32) ring(std::integral_constant<int, 2>{});
  else ring(std::integral_constant<int, TF>{});
  __syncthreads();   // every wave is done with the ring: the sums meet in its place
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int t = 0; t < TF; ++t) red[(wave * RF * TF + r * TF + t) * 64 + lane] = acc[r][t];
  __syncthreads();
  for (int e = tid; e < (GATED ? RF * TF * 32 : RF * TF * 64); e += 64 * WV) {   // 4 neighbouring columns of one row
    int f = e >> 6, l = e & 63, f2 = 0, l2 = 0;
    if constexpr (GATED) {   // ROWS 16: both halves in one operand, 32 lanes apart
      if constexpr (RF == 1) { f = e >> 5; l = e & 31; f2 = f; l2 = l + 32; }
      else { f2 = f + RF / 2 * TF; l2 = l; }
    }
    const int t = (f % TF) * 16 + (l & 15), n = n0 + (f / TF) * 16 + (l >> 4) * 4;
    if (t >= count || (ROWS == 8 && l >= 32)) continue;
    auto sum = [&](int ff, int ll) {
      f32x4_t v = red[ff * 64 + ll];
#pragma unroll
      for (int i = 1; i < WV; ++i) v += red[(i * RF * TF + ff) * 64 + ll];
      return v;
    };
    if constexpr (GATED) lin_gated4(a, lo + t, n, sum(f, l), sum(f2, l2), vec4);
    else lin_epilogue4<!SEG>(a, g, lo + t, n, sum(f, l), lin_bias4(a, g, n, vec4), vec4);
  }
}
template <int ROWS, int TF, bool SEG, bool GATED>
int launch_stream_lds_tf(const LinArgs& a, int groups, hipStream_t s) {
  // two workgroups per CU where two blocks per wave fit half of its LDS, else one
  constexpr int WV = STREAM_LDS_WAVES, PER = ROWS / 8 + 2 * TF, LDS_KB = ROWS < 64 && WV * 2 * PER <= 80 ? 80 : 160;
  constexpr int BY_LDS = LDS_KB / (WV * PER), BY_COUNT = 63 / PER + 1, D = BY_LDS < BY_COUNT ? BY_LDS : BY_COUNT, LDS = WV * D * PER * 1024;
  static_assert(D >= 2 && LDS >= WV * ((ROWS + 15) / 16) * TF * 1024, "two blocks, and room for the sums");
  auto kern = linear_stream_lds_kernel<ROWS, TF, WV, D, SEG, GATED>;
  if (LDS > 64 * 1024)
    DIHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS), DIHIP_RUNTIME_ERROR);
  hipLaunchKernelGGL(kern, dim3(GATED ? (a.N + ROWS / 2 - 1) / (ROWS / 2) : (a.N + ROWS - 1) / ROWS, groups), dim3(64 * WV), LDS, s, a, lin_vec4(a));
  return launch_status();
}
template <int ROWS, bool SEG, bool GATED = false>
int launch_stream_lds(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const int tf = (Tg + 15) / 16;
  return tf <= 1 ? launch_stream_lds_tf<ROWS, 1, SEG, GATED>(a, groups, s) : tf == 2 ? launch_stream_lds_tf<ROWS, 2, SEG, GATED>(a, groups, s)
         : tf == 3 ? launch_stream_lds_tf<ROWS, 3, SEG, GATED>(a, groups, s) : launch_stream_lds_tf<ROWS, 4, SEG, GATED>(a, groups, s);
}
// weight rows per workgroup: more of them bring the activations less often, but the workgroups have to fill 256 CUs.  16 / 32 / 64, us: 24 rows 4096 -> 4096
// 11.1 / 13.6 / 17.1, 2048 -> 8192 11.4 / 10.6 / 13.0, 4096 -> 14336 30.5 / 29.3 / 25.7, 4096 -> 32000 61 / 58 / 58 (64 rows of x: 88 / 74 / 63); 2 rows, whose
// activations are cheap, 9.1 / 9.8 / 11.0, 23.7 / 27.4 / 24.8 and 47 / 56 / 55.  Up to 2048 columns, of which 16 a workgroup leave half of the CUs without one, 8 (in an operand
// that holds them twice): 8 / 16, us, weights from memory: 8192 -> 2048 2 rows 9.1 / 11.1, 24 rows 12.7 / 15.0, 64 rows 20.5 / 22.4; 2048 -> 2048 5.7 / 6.1 at 24 rows; 4096 -> 1024
// 7.6 / 8.6; but 2048 -> 3072 8.0 / 6.5.  9 .. 16 rows of 4096 and more: 16 / 32 / 64 at 13 rows 4096 -> 8192 16.1 / 17.3 / 17.7, 4096 -> 32000 51.0 / 55.9 / 55.9, but 2048 -> 6208
// 8.7 / 8.2 / 10.0.  24 rows 4096 -> 12352 29.1 / 27.9 / 24.7, 2048 -> 32000 33.1 / 31.1 / 32.5.  Four waves in each form: an element's sum is the same in all of them.
// Segments hold few rows each, whatever the bound: 16 / 32 / 64 at 2048 -> 2816 of 64 experts, 6 per token, 4 tokens 49.3 / 50.9 / 56.0, 48 tokens 135.8 / 135.6 /
// 143.4; 2048 -> 4096 of 32, 4 per token, 4 tokens 45.7 / 43.1 / 41.4; 4096 -> 4096 of 32, 3 tokens 65.9 / 79.4 / 73.8, 48 tokens 183 / 205 / 210; 64 tokens through 2048 -> 2816
// 138.6 / 154.9 / 149.9 (four row operands leave the 32 form one workgroup per CU).
inline int launch_stream_lds_rows(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const long n = (long)a.N * groups;
  if (a.seg) return a.K < 4096 && Tg <= 48 ? launch_stream_lds<32, true>(a, Tg, groups, s) : launch_stream_lds<16, true>(a, Tg, groups, s);
  if (n <= 2048) return launch_stream_lds<8, false>(a, Tg, groups, s);
  if (n < 6144 || Tg <= (a.K >= 4096 ? 16 : 8)) return launch_stream_lds<16, false>(a, Tg, groups, s);
  return n < 12288 || (a.K <= 2048 && Tg <= 48) ? launch_stream_lds<32, false>(a, Tg, groups, s) : launch_stream_lds<64, false>(a, Tg, groups, s);
}

// The gated form has twice the weight rows of one product, so its lines lie elsewhere.  Two products / 16 / 32 / 64, us (weights from memory): 2048 -> 1408 24 rows 10.7 / 5.7 /
// 6.5 / 7.8; 1024 -> 3072 24 rows 9.3 / 6.3 / 5.7 / 6.3; 2048 -> 8192 13 rows 21.0 / 16.2 / 15.0 / 17.0, 24 rows 21.4 / 18.3 / 15.5 / 17.4, 64 rows 26.6 / 25.9 / 21.4 / 19.2; 4096 -> 6144
// 8 rows 27.8 / 20.6 / 23.3 / 23.9; 4096 -> 14336 13 rows 49.8 / 44.1 / 46.1 / 48.0, 24 rows 52.2 / 52.4 / 48.7 / 49.1, 64 rows 61.3 / 75.9 / 65.4 / 56.3.
inline int launch_stream_lds_gated(const LinArgs& a, hipStream_t s) {
  if (a.N < 3072 || (a.T <= 16 && a.K >= 4096)) return launch_stream_lds<16, false, true>(a, a.T, 1, s);
  return a.T <= 48 || a.N < 4096 ? launch_stream_lds<32, false, true>(a, a.T, 1, s) : launch_stream_lds<64, false, true>(a, a.T, 1, s);
}

template <int XT, int ROWS, int WV, bool PRE>
void launch_stream(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const dim3 grid((a.N + ROWS - 1) / ROWS, groups), threads(64 * WV);
  const int tf = (Tg + 15) / 16;
  const bool vec4 = lin_vec4(a);
  if (tf <= 1) hipLaunchKernelGGL((linear_stream_kernel<XT, ROWS, 1, WV, PRE>), grid, threads, 0, s, a, vec4);
  else if (tf == 2) hipLaunchKernelGGL((linear_stream_kernel<XT, ROWS, 2, WV, PRE>), grid, threads, 0, s, a, vec4);
  else if (tf == 3) hipLaunchKernelGGL((linear_stream_kernel<XT, ROWS, 3, WV, PRE>), grid, threads, 0, s, a, vec4);
  else hipLaunchKernelGGL((linear_stream_kernel<XT, ROWS, 4, WV, PRE>), grid, threads, 0, s, a, vec4);
}
// weight rows per workgroup: more of them re-read the activations less often, but the workgroups have to fill 256 CUs.  16 / 32 / 64 at
// 24 rows: 4096 -> 4096 15.1 / 18.8 / 28, 4096 -> 6144 25.0 / 22.4 / 24, 4096 -> 14336 43.1 / 40.9 / 36.9, 4096 -> 32000 106 / 84 / 69 us; at
// 4 rows the activations are cheap and 16 is never behind.  How many waves share K follows the width alone: an element's sum is the same for 2 rows and
// for 64.
template <int XT>
void launch_stream_rows(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const long n = (long)a.N * groups;
  if (n < 6144) launch_stream<XT, 16, 8, true>(a, Tg, groups, s);
  else if (Tg <= 8) launch_stream<XT, 16, 4, true>(a, Tg, groups, s);
  else if (Tg <= 16 || n < 16384) launch_stream<XT, 32, 4, true>(a, Tg, groups, s);
  else launch_stream<XT, 64, 4, false>(a, Tg, groups, s);
}

// ------------------------------------------------------------------------------------------ weight-streaming kernel
__device__ __forceinline__ float dot8_bf16(const u32x4_t& w, const u32x4_t& x, float acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc = __builtin_fmaf(__uint_as_float(w[i] << 16), __uint_as_float(x[i] << 16), acc);
    acc = __builtin_fmaf(__uint_as_float(w[i] & 0xffff0000u), __uint_as_float(x[i] & 0xffff0000u), acc);
  }
  return acc;
}

// One row of x (decoding one sequence) against bf16 weights.  Bound by the weights' bytes, in launches too short for workgroups that come and go: two
// workgroups per CU live for the whole launch, each owns a run of neighbouring weight rows, its 4 waves hold a quarter of x each -- C pieces of
// 512 elements, in registers as f32 -- and walk the same weight rows, so that the loop is weight loads and multiply-adds and nothing else.  Two batches of
// about 8 KiB per wave in turn, the next in flight while one is multiplied (copying one into the other would wait for it).
// The sums of the waves meet in LDS once, at the end; a lane's k ascend, lanes and waves are added in a fixed order.
// One wave per two weight rows (linear_skinny_kernel) -> this, us: 4096 -> 4096 11.5 -> 8.0, 14336 -> 4096 29.4 -> 21.7, 4096 -> 14336 26.9 -> 21.8,
// 4096 -> 32000 52.7 -> 44.5 (5.9 TB/s).
// MASK: K does not fill the pieces: the loads stay inside the row, and both x and the weights are zero past K (either may hold an infinity where it is re-read).
constexpr int ROW_WAVES = 4, ROW_WGS = 512, ROW_MAXC = 8, ROW_MAX_ROWS = 1024;   // weight rows of a workgroup: 16 KB of sums
// GATED: the rows of w that a workgroup owns, then the same ones of w2.  4096 -> 14336 twice 39.9 -> 35.1 us.
template <int XT, int C, bool MASK, bool GATED>
__global__ __launch_bounds__(64 * ROW_WAVES, 2) void linear_row_kernel(LinArgs a) {
  constexpr int R = C >= 5 ? 1 : 8 / C;        // weight rows per batch
  extern __shared__ __attribute__((aligned(16))) float part[];   // [row][wave]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = (int)((long)a.N * blockIdx.x / gridDim.x), hi = (int)((long)a.N * (blockIdx.x + 1) / gridDim.x);
  const uint16_t* w = (const uint16_t*)a.w + (size_t)lo * a.K;
  const uint16_t* w2 = GATED ? (const uint16_t*)a.w2 + (size_t)lo * a.K : nullptr;
  int k[C];
#pragma unroll
  for (int c = 0; c < C; ++c) k[c] = ((wave * C + c) * 64 + lane) * 8;
  const int own = hi - lo, rows = GATED ? 2 * own : own;
  auto load = [&](u32x4_t (&d)[R][C], int r0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = min(r0 + r, rows - 1);   // (uniform) past the end: the last row once more
      const uint16_t* row = GATED && i >= own ? w2 + (size_t)(i - own) * a.K : w + (size_t)i * a.K;
#pragma unroll
      for (int c = 0; c < C; ++c) d[r][c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(row + (MASK ? min(k[c], a.K - 8) : k[c])));
    }
  };
  u32x4_t wa[R][C], wb[R][C], q[C], q2[C];   // (q2: f32 rows)
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const size_t src = lin_xrow(a, 0) * a.ldx + (MASK ? min(k[c], a.K - 8) : k[c]);
    q[c] = *reinterpret_cast<const u32x4_t*>((const unsigned char*)a.x + src * (XT == DIHIP_F32 ? 4 : 2));
    if constexpr (XT == DIHIP_F32) q2[c] = *reinterpret_cast<const u32x4_t*>((const float*)a.x + src + 4);
  }
  load(wa, 0);
  __builtin_amdgcn_sched_barrier(0);
  float x[C][8];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if constexpr (XT == DIHIP_F32) {
      const f32x4_t l4 = __builtin_bit_cast(f32x4_t, q[c]), h4 = __builtin_bit_cast(f32x4_t, q2[c]);
      q[c] = u32x4_t{pack_bf16x2(l4[0], l4[1]), pack_bf16x2(l4[2], l4[3]), pack_bf16x2(h4[0], h4[1]), pack_bf16x2(h4[2], h4[3])};
    }
    if (MASK && k[c] >= a.K) q[c] = u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[c][2 * i] = __uint_as_float(q[c][i] << 16);
      x[c][2 * i + 1] = __uint_as_float(q[c][i] & 0xffff0000u);
    }
  }
  auto mul = [&](u32x4_t (&d)[R][C], int r0) {
    float v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] = 0.f;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (MASK && k[c] >= a.K) d[r][c] = u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[r] = __builtin_fmaf(__uint_as_float(d[r][c][i] << 16), x[c][2 * i], v[r]);
          v[r] = __builtin_fmaf(__uint_as_float(d[r][c][i] & 0xffff0000u), x[c][2 * i + 1], v[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = wave_sum(v[r]);
    if (lane == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r0 + r < rows) part[(r0 + r) * ROW_WAVES + wave] = v[r];
    }
  };
  LinRes res{0.f, 0.f, 0.f, 0.f};
  if (!GATED && a.res && tid < own) res = lin_res_load(a, 0, lo + tid);   // (a thread's first column: here long before it is used)
  for (int r0 = 0; r0 < rows; r0 += 2 * R) {
    load(wb, r0 + R);
    __builtin_amdgcn_sched_barrier(0);
    mul(wa, r0);
    __builtin_amdgcn_sched_barrier(0);
    load(wa, r0 + 2 * R);
    __builtin_amdgcn_sched_barrier(0);
    mul(wb, r0 + R);
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  for (int r = tid; r < own; r += 64 * ROW_WAVES) {
    const f32x4_t p = *reinterpret_cast<const f32x4_t*>(part + r * ROW_WAVES);
    const float v = (p[0] + p[1]) + (p[2] + p[3]);
    if constexpr (GATED) {
      const f32x4_t u = *reinterpret_cast<const f32x4_t*>(part + (own + r) * ROW_WAVES);
      st_any(a.y, (size_t)(lo + r), a.ydt, apply_act(v, a.act) * ((u[0] + u[1]) + (u[2] + u[3])));
    } else if (a.res && r == tid && !a.bias && !a.mul && a.act_hi <= a.act_lo) {
      lin_res_store(a, 0, lo + r, v, res);
    } else {
      lin_epilogue(a, 0, 0, lo + r, v, DIHIP_BF16);
    }
  }
}
template <int XT, int C, bool GATED>
void launch_row_c(const LinArgs& a, hipStream_t s) {
  const int wgs = a.N < ROW_WGS ? a.N : ROW_WGS;
  const size_t lds = (size_t)((a.N + wgs - 1) / wgs) * ROW_WAVES * sizeof(float) * (GATED ? 2 : 1);
  if (a.K == C * 512 * ROW_WAVES) hipLaunchKernelGGL((linear_row_kernel<XT, C, false, GATED>), dim3(wgs), dim3(64 * ROW_WAVES), lds, s, a);
  else hipLaunchKernelGGL((linear_row_kernel<XT, C, true, GATED>), dim3(wgs), dim3(64 * ROW_WAVES), lds, s, a);
}
inline int row_pieces(int K) { return (K + 512 * ROW_WAVES - 1) / (512 * ROW_WAVES); }
// where it is the faster one: long rows always, rows of 1024 .. 2048 from 12 MB of weights on.  linear_skinny_kernel / this, us: 64 x 4096 5.4 / 3.6,
// 1000 x 2560 5.5 / 5.1, 4096 x 1536 6.2 / 6.0, 8192 x 1024 7.1 / 5.9; but 2048 x 2048 5.3 / 5.6, 4096 x 1024 4.9 / 5.4, 100000 x 256 25.2 / 29.2
// (waves without a piece)
inline bool row_kernel(int N, int K) {
  return row_pieces(K) <= ROW_MAXC && (N + ROW_WGS - 1) / ROW_WGS <= ROW_MAX_ROWS && (K > 2048 || (K >= 1024 && (long)N * K >= 6000000));
}
template <int XT, bool GATED = false>
void launch_row(const LinArgs& a, hipStream_t s) {
  switch (row_pieces(a.K)) {
    case 1: return launch_row_c<XT, 1, GATED>(a, s);
    case 2: return launch_row_c<XT, 2, GATED>(a, s);
    case 3: return launch_row_c<XT, 3, GATED>(a, s);
    case 4: return launch_row_c<XT, 4, GATED>(a, s);
    case 5: return launch_row_c<XT, 5, GATED>(a, s);
    case 6: return launch_row_c<XT, 6, GATED>(a, s);
    case 7: return launch_row_c<XT, 7, GATED>(a, s);
    default: return launch_row_c<XT, 8, GATED>(a, s);
  }
}

// rows t0 .. t0 + tc (tc <= 4) of x staged in LDS -- as bf16, or as they are (EXACT: f32 products of the unrounded row) --;
// wave w of block b owns weight rows (b * 4 + w) * 2 .. + 2 and keeps two 1 KiB slices of each in flight.
// K % 8 == 0 and 16-byte aligned weight rows (host-checked).
template <int XT, bool EXACT>
__global__ __launch_bounds__(256) void linear_skinny_kernel(LinArgs a, int t0, int tc) {
  if (a.seg) {   // rows t0 .. of the group's own segment (block-uniform)
    const int lo = a.seg[blockIdx.y] + t0, left = a.seg[blockIdx.y + 1] - lo;
    if (left <= 0) return;
    t0 = lo;
    tc = min(tc, left);
  }
  extern __shared__ __attribute__((aligned(16))) unsigned char xraw[];
  uint16_t* xsm = reinterpret_cast<uint16_t*>(xraw);
  float* xsf = reinterpret_cast<float*>(xraw);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.y;
  const size_t xoff = (size_t)(g % a.xgroups) * a.xg;
  const int nb = (blockIdx.x * 4 + wave) * 2;
  const bool mine = nb < a.N;
  const uint16_t* wp = (const uint16_t*)a.w + (size_t)g * a.N * a.K;
  const uint16_t* w0 = wp + (size_t)min(nb, a.N - 1) * a.K;
  const uint16_t* w1 = wp + (size_t)min(nb + 1, a.N - 1) * a.K;
  const u32x4_t z = {0u, 0u, 0u, 0u};
  u32x4_t cur[2][2], nxt[2][2];
  auto wload = [&](u32x4_t (&d)[2][2], int k) {   // two 1 KiB slices of both rows, zeros beyond K
    const bool one = k < a.K, two = k + 512 < a.K;
    d[0][0] = one ? *reinterpret_cast<const u32x4_t*>(w0 + k) : z;
    d[1][0] = one ? *reinterpret_cast<const u32x4_t*>(w1 + k) : z;
    d[0][1] = two ? *reinterpret_cast<const u32x4_t*>(w0 + k + 512) : z;
    d[1][1] = two ? *reinterpret_cast<const u32x4_t*>(w1 + k + 512) : z;
  };
  wload(cur, lane * 8);     // in flight while the rows are staged
  // staging in units of 8 elements (K % 8 == 0, 16-byte aligned rows: host-checked), several units of a thread in flight
  const int upr = a.K >> 3, units = tc * upr;
#pragma unroll 4
  for (int u = tid; u < units; u += 256) {
    const int t = u / upr, k = (u - t * upr) * 8;
    const size_t src = lin_xrow(a, t0 + t) * a.ldx + xoff + k;
    float v[8];
    if constexpr (XT == DIHIP_F32) {
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>((const float*)a.x + src);
      const f32x4_t hi = *reinterpret_cast<const f32x4_t*>((const float*)a.x + src + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) { v[j] = lo[j]; v[4 + j] = hi[j]; }
    } else {
      const u32x4_t r = *reinterpret_cast<const u32x4_t*>((const uint16_t*)a.x + src);
#pragma unroll
      for (int j = 0; j < 4; ++j) { v[2 * j] = __uint_as_float(r[j] << 16); v[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u); }
    }
    if constexpr (EXACT) {
      *reinterpret_cast<f32x4_t*>(xsf + (size_t)t * a.K + k) = f32x4_t{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<f32x4_t*>(xsf + (size_t)t * a.K + k + 4) = f32x4_t{v[4], v[5], v[6], v[7]};
    } else {
      *reinterpret_cast<u32x4_t*>(xsm + (size_t)t * a.K + k) =
          u32x4_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    }
  }
  __syncthreads();
  if (!mine) return;
  float acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[i][t] = 0.f;
  for (int k = lane * 8; k < a.K; k += 1024) {
    wload(nxt, k + 1024);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kk = k + h * 512;
      if (kk >= a.K) break;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t < tc) {
          if constexpr (EXACT) {
            const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(xsf + (size_t)t * a.K + kk);
            const f32x4_t hi = *reinterpret_cast<const f32x4_t*>(xsf + (size_t)t * a.K + kk + 4);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              float v = acc[i][t];
              v = __builtin_fmaf(__uint_as_float(cur[i][h][0] << 16), lo[0], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][0] & 0xffff0000u), lo[1], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][1] << 16), lo[2], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][1] & 0xffff0000u), lo[3], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][2] << 16), hi[0], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][2] & 0xffff0000u), hi[1], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][3] << 16), hi[2], v);
              v = __builtin_fmaf(__uint_as_float(cur[i][h][3] & 0xffff0000u), hi[3], v);
              acc[i][t] = v;
            }
          } else {
            const u32x4_t xv = *reinterpret_cast<const u32x4_t*>(xsm + (size_t)t * a.K + kk);
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[i][t] = dot8_bf16(cur[i][h], xv, acc[i][t]);
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) cur[i][h] = nxt[i][h];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float v = wave_sum(acc[i][t]);
      if (lane == 0 && t < tc && nb + i < a.N) lin_epilogue(a, g, t0 + t, nb + i, v, DIHIP_BF16);
    }
}

// Where 2 .. 4 rows that cannot stream through LDS (f32 rows, K % 64 != 0) are faster here than in linear_stream_kernel: wide matrices, whose weights are all that
// counts and which have more than one workgroup of 16 columns per CU there; narrow ones, which leave CUs without one; and a K whose blocks of 128 do not fall evenly on
// 4 or 8 waves.  Against it: each further row costs it dot products (5 rows take two passes: 1.1 .. 2 times as long), rows of a power of two are its slowest, and below
// K = 896 there is little to stream.  This / linear_stream_kernel, us, f32 rows: 2 rows 4096 -> 16384 31.6 / 33.1, 4096 -> 64 6.9 / 8.5, 2048 -> 4608 8.0 / 10.7, 4104 -> 6144
// 16.1 / 24.1, 1000 -> 24000 13.9 / 20.8, 5120 -> 1024 9.4 / 12.1; 4 rows 2560 -> 50000 44.6 / 71.7, 4096 -> 32000 54.6 / 65.0, 1024 -> 128256 51.7 / 66.3; but 2 rows 4096 -> 4096
// 12.6 / 11.5, 2048 -> 8192 12.2 / 11.6, 512 -> 32000 13.0 / 10.8, 4 rows 8192 -> 8192 44.7 / 35.5.  Over 957 products of 2 .. 4 rows, 328 .. 8192 -> 64 .. 128256, the
// choice is on average 0.4 % behind the faster of both, and 18 are more than 3 % behind this kernel, at worst by 9 % (in a second session 4 rows 8192 -> 64 by 13 %, 1.9 us).
// Segments hold a row or two of up to 16 tokens, and the other kernel multiplies for the bound: 3 tokens, 2 of 16 experts 2048 -> 1408 10.7 / 16.2; 8 tokens, 8 of 128 experts
// 2048 -> 1536 63 / 75; 16 tokens, 4 of 32 experts 2880 -> 2880 98 / 117; but 6 tokens, 2 of 8 experts 1024 -> 2048 14.0 / 11.3, 16 tokens, 6 of 64 experts 2048 -> 2816 0.93 of it.
inline bool skinny_rows(int T, int N, int groups, int K, bool seg) {
  if (seg) return T <= 4 || (T <= 8 && (groups >= 16 || (groups >= 8 && K >= 2048 && K <= 8192))) || (T <= 16 && K % 128 != 0 && groups >= 32);
  if (T > 4 || K < 896) return false;
  const long n = (long)N * groups;
  const bool even = (K & (K - 1)) == 0, wide = n > 4096, mid = wide && n < 6144;
  if (even && T < 4 && n >= 8192 && n < 12288) return false;   // (512 workgroups there: two per CU)
  if (T == 2) return wide || n <= 1024 || (K >= 2048 && n <= 1536) || (K >= 2560 && !even);
  if (T == 3)
    return (K >= 2048 && n <= 512) || (K >= 2560 && !even && n <= 2048) || (wide && (K >= 2560 || mid || K % 128 != 0)) || (K >= 1536 && n >= 20000) || n >= 50000;
  return (wide && K >= 2560 && !even) || (mid && K >= 1536) || (K <= 4096 && (n >= 32000 || (n >= 20000 && K % 128 != 0)));
}
// Segments of 17 .. 64 tokens whose rows cannot stream through LDS: where the tiles of linear_mfma_kernel, which skip the row blocks a segment does not have, are faster than
// linear_stream_kernel, which multiplies for the bound.  This / that, us: 4 of 32 experts 2880 -> 2880, 64 tokens 135 / 182; 6 of 64, 2056 -> 2816, 33 tokens 1 / 1.36; 2048 -> 2816 64
// tokens 193 / 226, but 48 tokens 1 / 0.97; 8 of 256, 1024 -> 512, 24 tokens 39 / 47, 48 tokens 1 / 0.87; 2 of 16, 1408 -> 2048, 64 tokens 1 / 0.61.
inline bool seg_in_tiles(int T, int groups, int K) {
  return T > 16 && ((K % 128 != 0 && groups >= 32) || (T <= 32 && groups >= 256) || (T > 48 && (groups >= 64 || (K >= 2048 && K <= 8192 && (K & (K - 1)) != 0))));
}

// Few output columns against many rows (a router's logits): one workgroup per row, the row staged in LDS as f32, a wave per
// column: f32 products of the unrounded row, each lane over its k in ascending order, then the fixed tree over the lanes.
// K % 8 == 0 and 16-byte aligned weight rows (host-checked).
template <int XT>
__global__ __launch_bounds__(256) void linear_fewcols_kernel(LinArgs a) {
  extern __shared__ __attribute__((aligned(16))) float xrow[];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int k = tid; k < a.K; k += 256) xrow[k] = load_ft<XT>(a.x, (size_t)t * a.ldx + k);
  __syncthreads();
  for (int n = wave; n < a.N; n += 4) {
    const uint16_t* wr = (const uint16_t*)a.w + (size_t)n * a.K;
    float acc = 0.f;
    for (int k = lane * 8; k < a.K; k += 512) {
      const u32x4_t wv = *reinterpret_cast<const u32x4_t*>(wr + k);
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(xrow + k), hi = *reinterpret_cast<const f32x4_t*>(xrow + k + 4);
      acc = __builtin_fmaf(__uint_as_float(wv[0] << 16), lo[0], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[0] & 0xffff0000u), lo[1], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[1] << 16), lo[2], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[1] & 0xffff0000u), lo[3], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[2] << 16), hi[0], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[2] & 0xffff0000u), hi[1], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[3] << 16), hi[2], acc);
      acc = __builtin_fmaf(__uint_as_float(wv[3] & 0xffff0000u), hi[3], acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) lin_epilogue<false>(a, 0, t, n, acc, DIHIP_BF16);
  }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace dihip

using namespace dihip;

static int linear_impl(void* stream, const void* x, int x_dtype, long ldx, long x_gstride, int x_groups, const void* w,
                       int w_dtype, const void* bias, void* y, int y_dtype, long ldy, long y_gstride, const float* mul,
                       long ldm, int mul_group, int T, int N, int K, int groups, int act, int act_lo, int act_hi, float act_param, int math,
                       const int32_t* seg, const int32_t* row_map, int seg_max_rows, void* ws, size_t ws_bytes, const LinArgs* res = nullptr) {
  DIHIP_REQUIRE(T >= 0 && N > 0 && K > 0 && groups > 0 && x_groups > 0, DIHIP_PARAM_ERROR, "linear: bad shape T %d N %d K %d groups %d", T, N, K, groups);
  DIHIP_REQUIRE(seq_dtype_ok(x_dtype) && seq_dtype_ok(w_dtype) && seq_dtype_ok(y_dtype), DIHIP_PARAM_ERROR, "linear: f32 / bf16 only");
  DIHIP_REQUIRE(x && w && y, DIHIP_PARAM_ERROR, "linear: null pointer");
  DIHIP_REQUIRE(ldx >= K && ldy >= N && (!mul || ldm >= (mul_group ? groups : N)), DIHIP_PARAM_ERROR, "linear: a row stride below the row length");
  DIHIP_REQUIRE(math == DIHIP_MATH_F32 || math == DIHIP_MATH_BF16 || math == DIHIP_MATH_F32_STREAM, DIHIP_PARAM_ERROR,
                "linear: unknown math mode %d", math);
  DIHIP_REQUIRE(groups <= 65535, DIHIP_PARAM_ERROR, "linear: more than 65535 groups");
  DIHIP_REQUIRE(act != DIHIP_SEQ_ACT_SOFTCAP || act_param > 0.f, DIHIP_PARAM_ERROR, "linear: a cap must be positive");
  if (T == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  LinArgs a{x, ldx, x_gstride, x_groups, w, bias, y, ldy, y_gstride, mul, ldm, T, N, K, act, act_lo, act_hi, y_dtype, 0, mul_group, act_param, seg, row_map};
  if (res) {
    a.res = 1; a.res_a = res->res_a; a.res_lda = res->res_lda;
    a.norm_alpha = res->norm_alpha; a.norm_w = res->norm_w; a.norm_b = res->norm_b; a.h16 = res->h16;
  }
  const int Tg = seg ? (seg_max_rows < T ? seg_max_rows : T) : T;   // the most rows one group can have
  const size_t xe = x_dtype == DIHIP_F32 ? 4 : 2;
  const bool vec = w_dtype == DIHIP_BF16 && K % 8 == 0 && aligned16(w) && aligned16(x) && (ldx * xe) % 16 == 0 &&
                   (x_gstride * xe) % 16 == 0;
  static const bool no_skinny = env_off("DIHIP_LINEAR_SKINNY");
  if (math == DIHIP_MATH_F32_STREAM) {
    // f32 products of unrounded rows; few rows stream the weight once (a row's sum then runs in the lanes' order, not k ascending)
    const int tmax = K <= 4096 ? 4 : (K <= 8192 ? 2 : 1);
    if (Tg <= 4 * tmax && vec && !no_skinny && K <= 16384) {
      for (int t0 = 0; t0 < Tg; t0 += tmax) {
        const int tc = Tg - t0 < tmax ? Tg - t0 : tmax;
        const dim3 grid((N + 7) / 8, groups);
        if (x_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_skinny_kernel<DIHIP_F32, true>), grid, dim3(256), (size_t)tc * K * 4, s, a, t0, tc);
        else hipLaunchKernelGGL((linear_skinny_kernel<DIHIP_BF16, true>), grid, dim3(256), (size_t)tc * K * 4, s, a, t0, tc);
      }
      return launch_status();
    }
    if (N <= 64 && groups == 1 && !seg && vec && K <= 16384) {   // many rows, few columns: the tile kernel would idle most of its 64 x 64 tile
      if (x_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_fewcols_kernel<DIHIP_F32>), dim3(T), dim3(256), (size_t)K * 4, s, a);
      else hipLaunchKernelGGL((linear_fewcols_kernel<DIHIP_BF16>), dim3(T), dim3(256), (size_t)K * 4, s, a);
      return launch_status();
    }
    math = DIHIP_MATH_F32;
  }
  if (math == DIHIP_MATH_BF16 && w_dtype == DIHIP_BF16) {
    if (Tg == 1 && groups == 1 && !seg && vec && !no_skinny && row_kernel(N, K)) {
      if (x_dtype == DIHIP_F32) launch_row<DIHIP_F32>(a, s);
      else launch_row<DIHIP_BF16>(a, s);
      return launch_status();
    }
    const bool by_lds = Tg > 1 && Tg <= STREAM_MAX_ROWS && vec && x_dtype == DIHIP_BF16 && K % 64 == 0 && K >= (seg ? 512 : 1024) &&
                        (size_t)64 * K * 2 < (1ull << 31) && (seg || (size_t)T * ldx * 2 < (1ull << 31));   // (32-bit offsets but for segments)
    const int tmax = Tg < 4 ? Tg : 4;   // rows of a pass; their bf16 copies fit 64 KB of LDS
    if ((Tg == 1 || (!by_lds && skinny_rows(Tg, N, groups, K, seg != nullptr))) && vec && !no_skinny && (size_t)tmax * K * 2 <= 65536) {
      const dim3 grid((N + 7) / 8, groups);
      for (int t0 = 0; t0 < Tg; t0 += tmax) {
        const int tc = Tg - t0 < tmax ? Tg - t0 : tmax;
        if (x_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_skinny_kernel<DIHIP_F32, false>), grid, dim3(256), (size_t)tc * K * 2, s, a, t0, tc);
        else hipLaunchKernelGGL((linear_skinny_kernel<DIHIP_BF16, false>), grid, dim3(256), (size_t)tc * K * 2, s, a, t0, tc);
      }
      return launch_status();
    }
    if (by_lds) return launch_stream_lds_rows(a, Tg, groups, s);
    if (Tg <= STREAM_MAX_ROWS && vec && !(seg && (x_dtype == DIHIP_F32 || K % 64 != 0) && seg_in_tiles(Tg, groups, K))) {
      if (x_dtype == DIHIP_F32) launch_stream_rows<DIHIP_F32>(a, Tg, groups, s);
      else launch_stream_rows<DIHIP_BF16>(a, Tg, groups, s);
      return launch_status();
    }
    if (vec && x_dtype == DIHIP_BF16) {
      // (segments: planned for twice the average, the bound is often all rows)
      const int rows = seg ? (int)std::min<long>(Tg, 1 + 2L * T / groups) : Tg;
      LinTilePlan p = plan_linear_tile(rows, N, K, groups, ldx, !seg && ws);
      if (p.ok && p.slab > ws_bytes) p = plan_linear_tile(rows, N, K, groups, ldx, false);
      if (p.ok) return launch_linear_tile(a, p, Tg, groups, (float*)ws, s);
    }
    const dim3 grid((N + 127) / 128, (Tg + 127) / 128, groups);
    DIHIP_REQUIRE(grid.y <= 65535, DIHIP_PARAM_ERROR, "linear: too many rows for one launch");
    const bool vec4 = lin_vec4(a);
    if (x_dtype == DIHIP_F32) {
      if (vec) hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_F32, true, false>), grid, dim3(256), 0, s, a, vec4);
      else hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_F32, false, false>), grid, dim3(256), 0, s, a, vec4);
    } else if (a.res) {
      if (vec) hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_BF16, true, true>), grid, dim3(256), 0, s, a, vec4);
      else hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_BF16, false, true>), grid, dim3(256), 0, s, a, vec4);
    } else {
      if (vec) hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_BF16, true, false>), grid, dim3(256), 0, s, a, vec4);
      else hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_BF16, false, false>), grid, dim3(256), 0, s, a, vec4);
    }
    return launch_status();
  }
  a.round_ops = math == DIHIP_MATH_BF16;
  const dim3 grid((N + 63) / 64, (Tg + 63) / 64, groups);
  DIHIP_REQUIRE(grid.y <= 65535, DIHIP_PARAM_ERROR, "linear: too many rows for one launch");
  if (x_dtype == DIHIP_F32 && w_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_tile_kernel<DIHIP_F32, DIHIP_F32>), grid, dim3(256), 0, s, a);
  else if (x_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_tile_kernel<DIHIP_F32, DIHIP_BF16>), grid, dim3(256), 0, s, a);
  else if (w_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_tile_kernel<DIHIP_BF16, DIHIP_F32>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((linear_tile_kernel<DIHIP_BF16, DIHIP_BF16>), grid, dim3(256), 0, s, a);
  return launch_status();
}

extern "C" int dihip_linear(void* stream, const void* x, int x_dtype, long ldx, long x_gstride, int x_groups, const void* w,
                            int w_dtype, const void* bias, void* y, int y_dtype, long ldy, long y_gstride, const float* mul,
                            long ldm, int mul_group, int T, int N, int K, int groups, int act, int act_lo, int act_hi,
                            float act_param, int math) {
  return linear_impl(stream, x, x_dtype, ldx, x_gstride, x_groups, w, w_dtype, bias, y, y_dtype, ldy, y_gstride, mul, ldm, mul_group, T, N, K, groups,
                     act, act_lo, act_hi, act_param, math, nullptr, nullptr, 0, nullptr, 0);
}

// Where the gated form runs as one launch: where each of its two products would take a kernel that has one
static bool gated_as_one(int T, int N, int K, long ldx) {
  static const bool no_skinny = env_off("DIHIP_LINEAR_SKINNY");
  if (T < 1 || N < 1 || K < 1 || K % 8 != 0 || ldx < K || ldx % 8 != 0) return false;
  if (T == 1) return !no_skinny && row_kernel(2 * N, K);
  if (T <= STREAM_MAX_ROWS) return K % 64 == 0 && K >= 1024 && (size_t)64 * K * 2 < (1ull << 31) && (size_t)T * ldx * 2 < (1ull << 31);
  return plan_linear_tile(T, N, K, 1, ldx, false, true).ok;
}

extern "C" int dihip_linear_gated_query(int T, int N, int K, long ldx, size_t* ws_bytes) {
  if (N > INT32_MAX / 2 || !gated_as_one(T, N, K, ldx)) return 0;
  *ws_bytes = T > STREAM_MAX_ROWS ? plan_linear_tile(T, N, K, 1, ldx, true, true).slab : 0;
  return 1;
}

extern "C" int dihip_linear_gated(void* stream, const void* x, long ldx, const void* w_gate, const void* w_up, void* y, int y_dtype, long ldy, int T, int N, int K,
                                  int act, void* ws, size_t ws_bytes) {
  DIHIP_REQUIRE(T >= 0 && N > 0 && N <= INT32_MAX / 2 && K > 0, DIHIP_PARAM_ERROR, "linear_gated: bad shape T %d N %d K %d", T, N, K);
  DIHIP_REQUIRE(x && w_gate && w_up && y && seq_dtype_ok(y_dtype) && ldy >= N && ldx >= K, DIHIP_PARAM_ERROR, "linear_gated: bad argument");
  DIHIP_REQUIRE(act >= 0 && act != DIHIP_SEQ_ACT_SOFTCAP, DIHIP_PARAM_ERROR, "linear_gated: no activation with a parameter");
  if (T == 0) return DIHIP_SUCCESS;
  DIHIP_REQUIRE(aligned16(x) && aligned16(w_gate) && aligned16(w_up) && (!ws || aligned16(ws)) && gated_as_one(T, N, K, ldx), DIHIP_EXCEED_LIMIT_ERROR,
                "linear_gated: T %d N %d K %d does not run as one launch", T, N, K);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  LinArgs a{};
  a.x = x; a.ldx = ldx; a.xgroups = 1; a.w = w_gate; a.w2 = w_up; a.y = y; a.ydt = y_dtype; a.ldy = ldy;
  a.T = T; a.N = N; a.K = K; a.act = act; a.act_hi = N;
  if (T == 1) {
    launch_row<DIHIP_BF16, true>(a, s);
    return launch_status();
  }
  if (T <= STREAM_MAX_ROWS) return launch_stream_lds_gated(a, s);
  LinTilePlan p = plan_linear_tile(T, N, K, 1, ldx, ws != nullptr, true);
  if (p.slab > ws_bytes) p = plan_linear_tile(T, N, K, 1, ldx, false, true);
  return launch_linear_tile(a, p, T, 1, (float*)ws, s);
}

extern "C" size_t dihip_linear_workspace_bytes(int T, int N, int K, int groups, long ldx) {
  if (T <= STREAM_MAX_ROWS || N <= 0 || K <= 0 || groups <= 0) return 0;
  return plan_linear_tile(T, N, K, groups, ldx, true).slab;
}

extern "C" int dihip_linear_ws(void* stream, const void* x, int x_dtype, long ldx, long x_gstride, int x_groups, const void* w,
                               int w_dtype, const void* bias, void* y, int y_dtype, long ldy, long y_gstride, const float* mul,
                               long ldm, int mul_group, int T, int N, int K, int groups, int act, int act_lo, int act_hi,
                               float act_param, int math, void* ws, size_t ws_bytes) {
  DIHIP_REQUIRE(!ws || aligned16(ws), DIHIP_PARAM_ERROR, "linear: a workspace starts on 16 bytes");
  return linear_impl(stream, x, x_dtype, ldx, x_gstride, x_groups, w, w_dtype, bias, y, y_dtype, ldy, y_gstride, mul, ldm, mul_group, T, N, K, groups,
                     act, act_lo, act_hi, act_param, math, nullptr, nullptr, 0, ws, ws_bytes);
}

extern "C" int dihip_linear_residual_dyt(void* stream, const void* x, long ldx, const void* w, float* stream_x, const float* a, long lda, float alpha, const void* norm_w,
                                         const void* norm_b, void* h16, int T, int N, int K, void* ws, size_t ws_bytes) {
  DIHIP_REQUIRE(!ws || aligned16(ws), DIHIP_PARAM_ERROR, "linear_residual_dyt: a workspace starts on 16 bytes");
  DIHIP_REQUIRE((!a || lda >= N) && (!norm_w || (norm_b && h16)), DIHIP_PARAM_ERROR, "linear_residual_dyt: bad argument");
  LinArgs r{};
  r.res_a = a; r.res_lda = lda; r.norm_alpha = alpha; r.norm_w = norm_w; r.norm_b = norm_w ? norm_b : nullptr; r.h16 = norm_w ? (uint16_t*)h16 : nullptr;
  return linear_impl(stream, x, DIHIP_BF16, ldx, K, 1, w, DIHIP_BF16, nullptr, stream_x, DIHIP_F32, N, N, nullptr, 0, 0, T, N, K, 1, 0, 0, 0, 0.f, DIHIP_MATH_BF16,
                     nullptr, nullptr, 0, ws, ws_bytes, &r);
}

extern "C" int dihip_linear_segmented(void* stream, const void* x, int x_dtype, long ldx, const void* w, int w_dtype, const void* bias,
                                      void* y, int y_dtype, long ldy, int R, int N, int K, int groups, const int32_t* seg,
                                      const int32_t* row_map, int seg_max_rows, int act, int math) {
  DIHIP_REQUIRE(seg && seg_max_rows >= 0, DIHIP_PARAM_ERROR, "linear_segmented: no segment table");
  if (seg_max_rows == 0) return DIHIP_SUCCESS;
  return linear_impl(stream, x, x_dtype, ldx, 0, 1, w, w_dtype, bias, y, y_dtype, ldy, 0, nullptr, 0, 0, R, N, K, groups, act, 0,
                     act ? groups * N : 0, 0.f, math, seg, row_map, seg_max_rows, nullptr, 0);
}
