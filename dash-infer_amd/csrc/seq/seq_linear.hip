// seq_linear.hip -- dihip_linear: y = epilogue(x . W^T + bias) for row-major [N, K] weights as checkpoints store them,
// grouped (block-diagonal / per-head) forms included.  The kernels:
//   linear_tile_kernel   every product and sum in f32, k ascending (DIHIP_MATH_F32; also any operand type / odd shape)
//   linear_pipe_kernel   bf16 operands on the matrix cores, pipelined tiles of 256 x 256 or 128 x 128, K split where tiles are few (seq_linear_tile.hip)
//   linear_mfma_kernel   the same for f32 rows (rounded to bf16), K % 64 != 0 or unaligned operands: 128 x 128 x 32 tiles through registers
//   linear_stream_lds_kernel  bf16 operands, 2 .. 64 rows, K % 64 == 0 and 1024 or more: both streamed through LDS, K split over a workgroup's waves
//   linear_stream_kernel the same for f32 rows, other K, gathered rows: weights straight from memory into the matrix cores
//   linear_row_kernel    one row (decode), bf16 operands: two workgroups per CU walk the weight rows past x in registers
//   linear_skinny_kernel one short row, one row per group, up to 4 rows at a time in f32 products: a streamed weight, one wave per 2 weight rows
//   linear_fewcols_kernel a router's logits
// Within a kernel an output element is summed over k in a fixed order: it does not depend on T.
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
      if (n < a.N) lin_epilogue(a, g, t, n, acc[i][j], WT);
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

template <int XT, bool VEC>
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
      if (t < t_hi) lin_epilogue4(a, g, t, n, acc[i][j], b, vec4);
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
constexpr int STREAM_LDS_WAVES = 4;
template <int ROWS, int TF, int WV, int D>
__global__ __launch_bounds__(64 * WV, 2) void linear_stream_lds_kernel(LinArgs a, bool vec4) {
  constexpr int RF = ROWS / 16, PER = 2 * (RF + TF), SLOT = PER * 1024;
  static_assert((D - 1) * PER < 64, "what is in flight is counted");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.y, n0 = blockIdx.x * ROWS;
  int lo, hi;
  lin_rows(a, g, lo, hi);
  if (lo >= hi) return;
  const int count = min(hi - lo, 16 * TF);
  const int prow = lane >> 3, pchunk = (lane & 7) ^ prow;
  const char* wbase = (const char*)((const uint16_t*)a.w + ((size_t)g * a.N + n0) * a.K);
  const char* xbase = (const char*)((const uint16_t*)a.x + (size_t)(g % a.xgroups) * a.xg);
  uint32_t off[PER];   // (the host checks that they fit); rows past N re-read the last one, rows past the group's the last of those: never stored
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int r = (p < 2 * RF ? p : p - 2 * RF) * 8 + prow;
    off[p] = p < 2 * RF ? (uint32_t)min(r, a.N - 1 - n0) * (uint32_t)a.K * 2 + pchunk * 16
                        : (uint32_t)(lin_xrow(a, lo + min(r, count - 1)) * a.ldx * 2) + pchunk * 16;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + wave * D * SLOT;
  const unsigned char* mine = lds + wave * D * SLOT;
  const int blocks = a.K / 64, steps = (blocks - wave + WV - 1) / WV;   // blocks wave, wave + WV, ..
  auto fetch = [&](int i, int slot) {
    const char* wk = wbase + (size_t)(wave + i * WV) * 128;
    const char* xk = xbase + (size_t)(wave + i * WV) * 128;
#pragma unroll
    for (int p = 0; p < PER; ++p)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + slot * SLOT + p * 1024), "v"(off[p]), "s"(p < 2 * RF ? wk : xk) : "memory");
  };
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[RF][TF];
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int t = 0; t < TF; ++t) acc[r][t] = z4;
  const int f0 = (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) * 16);
  auto mul = [&](int slot) {
    const unsigned char* b = mine + slot * SLOT;
    u32x4_t w[2][RF], x[2][TF];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < RF; ++r) w[h][r] = *reinterpret_cast<const u32x4_t*>(b + r * 2048 + (h ? f0 ^ 64 : f0));
#pragma unroll
      for (int t = 0; t < TF; ++t) x[h][t] = *reinterpret_cast<const u32x4_t*>(b + (RF + t) * 2048 + (h ? f0 ^ 64 : f0));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < RF; ++r)
#pragma unroll
        for (int t = 0; t < TF; ++t) acc[r][t] = mfma_bf16(w[h][r], x[h][t], acc[r][t]);
  };
  if (steps >= D) {
#pragma unroll
    for (int i = 0; i < D; ++i) fetch(i, i);
    int slot = 0;
    for (int i = 0; i + D < steps; ++i) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * PER) : "memory");
      mul(slot);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot has been read
      fetch(i + D, slot);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
#pragma unroll
    for (int j = 0; j < D; ++j) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1 - j) * PER) : "memory");
      mul(slot);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
  } else {
    for (int i = 0; i < steps; ++i) fetch(i, i);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    for (int i = 0; i < steps; ++i) mul(i);
  }
  __syncthreads();   // every wave is done with the ring: the sums meet in its place
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int t = 0; t < TF; ++t) red[(wave * RF * TF + r * TF + t) * 64 + lane] = acc[r][t];
  __syncthreads();
  for (int e = tid; e < RF * TF * 64; e += 64 * WV) {   // 4 neighbouring columns of one row
    const int f = e >> 6, l = e & 63, t = (f % TF) * 16 + (l & 15), n = n0 + (f / TF) * 16 + (l >> 4) * 4;
    if (t >= count) continue;
    f32x4_t v = red[f * 64 + l];
#pragma unroll
    for (int i = 1; i < WV; ++i) v += red[(i * RF * TF + f) * 64 + l];
    lin_epilogue4(a, g, lo + t, n, v, lin_bias4(a, g, n, vec4), vec4);
  }
}
template <int ROWS, int TF>
int launch_stream_lds_tf(const LinArgs& a, int groups, hipStream_t s) {
  // two workgroups per CU where two blocks per wave fit half of its LDS, else one
  constexpr int WV = STREAM_LDS_WAVES, PER = 2 * (ROWS / 16 + TF), LDS_KB = ROWS < 64 && WV * 2 * PER <= 80 ? 80 : 160;
  constexpr int BY_LDS = LDS_KB / (WV * PER), BY_COUNT = 63 / PER + 1, D = BY_LDS < BY_COUNT ? BY_LDS : BY_COUNT, LDS = WV * D * PER * 1024;
  static_assert(D >= 2 && LDS >= WV * (ROWS / 16) * TF * 1024, "two blocks, and room for the sums");
  auto kern = linear_stream_lds_kernel<ROWS, TF, WV, D>;
  if (LDS > 64 * 1024)
    DIHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS), DIHIP_RUNTIME_ERROR);
  hipLaunchKernelGGL(kern, dim3((a.N + ROWS - 1) / ROWS, groups), dim3(64 * WV), LDS, s, a, lin_vec4(a));
  return launch_status();
}
template <int ROWS>
int launch_stream_lds(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const int tf = (Tg + 15) / 16;
  return tf <= 1 ? launch_stream_lds_tf<ROWS, 1>(a, groups, s) : tf == 2 ? launch_stream_lds_tf<ROWS, 2>(a, groups, s)
         : tf == 3 ? launch_stream_lds_tf<ROWS, 3>(a, groups, s) : launch_stream_lds_tf<ROWS, 4>(a, groups, s);
}
// weight rows per workgroup: more of them bring the activations less often, but the workgroups have to fill 256 CUs.  16 / 32 / 64, us: 24 rows 4096 -> 4096
// 11.1 / 13.6 / 17.1, 2048 -> 8192 11.4 / 10.6 / 13.0, 4096 -> 14336 30.5 / 29.3 / 25.7, 4096 -> 32000 61 / 58 / 58 (64 rows of x: 88 / 74 / 63); 2 rows, whose
// activations are cheap, 9.1 / 9.8 / 11.0, 23.7 / 27.4 / 24.8 and 47 / 56 / 55.  Four waves in each form: an element's sum is the same in all of them.
inline int launch_stream_lds_rows(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const long n = (long)a.N * groups;
  if (n < 6144 || Tg <= 8) return launch_stream_lds<16>(a, Tg, groups, s);
  return n < 13312 ? launch_stream_lds<32>(a, Tg, groups, s) : launch_stream_lds<64>(a, Tg, groups, s);
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
// 4 rows the activations are cheap and 16 is never behind.
template <int XT>
void launch_stream_rows(const LinArgs& a, int Tg, int groups, hipStream_t s) {
  const long n = (long)a.N * groups;
  if (Tg > 16 && n >= 16384) launch_stream<XT, 64, 4, false>(a, Tg, groups, s);
  else if (Tg > 8 && n >= 6144) launch_stream<XT, 32, 4, true>(a, Tg, groups, s);
  else launch_stream<XT, 16, 8, true>(a, Tg, groups, s);
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
// MASK: K does not fill the pieces: x is zero there and the loads stay inside the row.
constexpr int ROW_WAVES = 4, ROW_WGS = 512, ROW_MAXC = 8, ROW_MAX_ROWS = 1024;   // weight rows of a workgroup: 16 KB of sums
template <int XT, int C, bool MASK>
__global__ __launch_bounds__(64 * ROW_WAVES, 2) void linear_row_kernel(LinArgs a) {
  constexpr int R = C >= 5 ? 1 : 8 / C;        // weight rows per batch
  extern __shared__ __attribute__((aligned(16))) float part[];   // [row][wave]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = (int)((long)a.N * blockIdx.x / gridDim.x), hi = (int)((long)a.N * (blockIdx.x + 1) / gridDim.x);
  const uint16_t* w = (const uint16_t*)a.w + (size_t)lo * a.K;
  int k[C];
#pragma unroll
  for (int c = 0; c < C; ++c) k[c] = ((wave * C + c) * 64 + lane) * 8;
  const int rows = hi - lo;
  auto load = [&](u32x4_t (&d)[R][C], int r0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint16_t* row = w + (size_t)min(r0 + r, rows - 1) * a.K;   // (uniform) past the end: the last row once more
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
  for (int r = tid; r < rows; r += 64 * ROW_WAVES) {
    const f32x4_t p = *reinterpret_cast<const f32x4_t*>(part + r * ROW_WAVES);
    lin_epilogue(a, 0, 0, lo + r, (p[0] + p[1]) + (p[2] + p[3]), DIHIP_BF16);
  }
}
template <int XT, int C>
void launch_row_c(const LinArgs& a, hipStream_t s) {
  const int wgs = a.N < ROW_WGS ? a.N : ROW_WGS;
  const size_t lds = (size_t)((a.N + wgs - 1) / wgs) * ROW_WAVES * sizeof(float);
  if (a.K == C * 512 * ROW_WAVES) hipLaunchKernelGGL((linear_row_kernel<XT, C, false>), dim3(wgs), dim3(64 * ROW_WAVES), lds, s, a);
  else hipLaunchKernelGGL((linear_row_kernel<XT, C, true>), dim3(wgs), dim3(64 * ROW_WAVES), lds, s, a);
}
inline int row_pieces(int K) { return (K + 512 * ROW_WAVES - 1) / (512 * ROW_WAVES); }
// where it is the faster one: long rows always, rows of 1024 .. 2048 from 12 MB of weights on.  linear_skinny_kernel / this, us: 64 x 4096 5.4 / 3.6,
// 1000 x 2560 5.5 / 5.1, 4096 x 1536 6.2 / 6.0, 8192 x 1024 7.1 / 5.9; but 2048 x 2048 5.3 / 5.6, 4096 x 1024 4.9 / 5.4, 100000 x 256 25.2 / 29.2
// (waves without a piece)
inline bool row_kernel(int N, int K) {
  return row_pieces(K) <= ROW_MAXC && (N + ROW_WGS - 1) / ROW_WGS <= ROW_MAX_ROWS && (K > 2048 || (K >= 1024 && (long)N * K >= 6000000));
}
template <int XT>
void launch_row(const LinArgs& a, hipStream_t s) {
  switch (row_pieces(a.K)) {
    case 1: return launch_row_c<XT, 1>(a, s);
    case 2: return launch_row_c<XT, 2>(a, s);
    case 3: return launch_row_c<XT, 3>(a, s);
    case 4: return launch_row_c<XT, 4>(a, s);
    case 5: return launch_row_c<XT, 5>(a, s);
    case 6: return launch_row_c<XT, 6>(a, s);
    case 7: return launch_row_c<XT, 7>(a, s);
    default: return launch_row_c<XT, 8>(a, s);
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
    if (lane == 0) lin_epilogue(a, 0, t, n, acc, DIHIP_BF16);
  }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace dihip

using namespace dihip;

static int linear_impl(void* stream, const void* x, int x_dtype, long ldx, long x_gstride, int x_groups, const void* w,
                       int w_dtype, const void* bias, void* y, int y_dtype, long ldy, long y_gstride, const float* mul,
                       long ldm, int mul_group, int T, int N, int K, int groups, int act, int act_lo, int act_hi, float act_param, int math,
                       const int32_t* seg, const int32_t* row_map, int seg_max_rows, void* ws, size_t ws_bytes) {
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
    if (Tg == 1 && vec && !no_skinny && K <= 32768) {   // the row's bf16 copy fits 64 KB of LDS
      const dim3 grid((N + 7) / 8, groups);
      if (x_dtype == DIHIP_F32) hipLaunchKernelGGL((linear_skinny_kernel<DIHIP_F32, false>), grid, dim3(256), (size_t)K * 2, s, a, 0, 1);
      else hipLaunchKernelGGL((linear_skinny_kernel<DIHIP_BF16, false>), grid, dim3(256), (size_t)K * 2, s, a, 0, 1);
      return launch_status();
    }
    if (Tg <= STREAM_MAX_ROWS && vec && x_dtype == DIHIP_BF16 && K % 64 == 0 && K >= 1024 && !row_map && (size_t)64 * K * 2 < (1ull << 31) &&
        (size_t)T * ldx * 2 < (1ull << 31))   // (32-bit offsets; a row map's targets are not known here)
      return launch_stream_lds_rows(a, Tg, groups, s);
    if (Tg <= STREAM_MAX_ROWS && vec) {
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
      if (vec) hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_F32, true>), grid, dim3(256), 0, s, a, vec4);
      else hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_F32, false>), grid, dim3(256), 0, s, a, vec4);
    } else {
      if (vec) hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_BF16, true>), grid, dim3(256), 0, s, a, vec4);
      else hipLaunchKernelGGL((linear_mfma_kernel<DIHIP_BF16, false>), grid, dim3(256), 0, s, a, vec4);
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

extern "C" int dihip_linear_segmented(void* stream, const void* x, int x_dtype, long ldx, const void* w, int w_dtype, const void* bias,
                                      void* y, int y_dtype, long ldy, int R, int N, int K, int groups, const int32_t* seg,
                                      const int32_t* row_map, int seg_max_rows, int act, int math) {
  DIHIP_REQUIRE(seg && seg_max_rows >= 0, DIHIP_PARAM_ERROR, "linear_segmented: no segment table");
  if (seg_max_rows == 0) return DIHIP_SUCCESS;
  return linear_impl(stream, x, x_dtype, ldx, 0, 1, w, w_dtype, bias, y, y_dtype, ldy, 0, nullptr, 0, 0, R, N, K, groups, act, 0,
                     act ? groups * N : 0, 0.f, math, seg, row_map, seg_max_rows, nullptr, 0);
}
