// glue.hip -- the bandwidth-trivial ops of a decode step (include/dashinfer_hip.h section 5):
// LayerNormNoBeta (RMSNorm), Rotary, Binary ADD, SiLU*MUL, greedy argmax, embedding lookup,
// device-side step counter.  All vectorised 16 B per lane where the layout allows.
#include <algorithm>

#include "device_utils.h"

namespace dihip {

// ---- LayerNormNoBeta: y = (gamma * x) * rsqrt(mean(x^2) + eps)  (layernorm.cpp:110-157) ------
template <int FT>
__global__ __launch_bounds__(256) void rmsnorm_kernel(void* __restrict__ y, const void* __restrict__ x,
                                                      const void* __restrict__ gamma, float eps, int cols) {
  __shared__ float red[4];
  const size_t row = (size_t)blockIdx.x * cols;
  float ss = 0.f;
  for (int k = threadIdx.x; k < cols; k += 256) {
    const float v = load_ft<FT>(x, row + k);
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float rstd = 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)cols + eps);
  for (int k = threadIdx.x; k < cols; k += 256)
    store_ft<FT>(y, row + k, (load_ft<FT>(gamma, k) * load_ft<FT>(x, row + k)) * rstd);
}

// ---- Rotary (rotate-half) on the q and k heads of fused qkv rows, in place ---------------------
// grid (rows, n + g), 64 lanes = H/2 pairs (H = 128) ; lanes >= H/2 idle for smaller heads
template <int FT>
__global__ __launch_bounds__(64) void rope_qk_kernel(void* qkv, const uint32_t* __restrict__ positions,
                                                     const float* __restrict__ inv_freq, int n, int g, int H) {
  const int row = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  const int half = H / 2;
  if (d >= half) return;
  const size_t base = (size_t)row * (n + 2 * g) * H + (size_t)head * H;  // q heads then k heads
  float sn, cs;
  rope_sincos(positions[row], inv_freq[d], &sn, &cs);
  const float x1 = load_ft<FT>(qkv, base + d), x2 = load_ft<FT>(qkv, base + d + half);
  store_ft<FT>(qkv, base + d, x1 * cs - x2 * sn);
  store_ft<FT>(qkv, base + d + half, x2 * cs + x1 * sn);
}

template <int FT, int OP>  // OP 0: a + b ; 1: silu(a) * b
__global__ __launch_bounds__(256) void binary_kernel(void* __restrict__ y, const void* __restrict__ a,
                                                     const void* __restrict__ b, size_t count) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t)gridDim.x * 256) {
    const float va = load_ft<FT>(a, i), vb = load_ft<FT>(b, i);
    float r;
    if constexpr (OP == 0) {
      r = va + vb;
    } else {
      // Gemm(gate) with fused SiLU produces an FT tensor, then Binary MUL (qwen_v15.py:314-335)
      float sa = va / (1.f + expf(-va));
      if constexpr (FT != DIHIP_F32) sa = ft_round<FT>(sa);
      r = sa * vb;
    }
    store_ft<FT>(y, i, r);
  }
}

// Binary MUL / Unary / UnaryGLU of the reference graph as stand-alone operators (csrc/core/kernel/cuda/binary.cu, unary.cu:120-133):
// the fused decode step never launches them (they ride in GEMV epilogues); the operator layer needs them so that an
// unmodified model graph resolves on DeviceType::HIP.  f32 arithmetic, one FT rounding of the result.
template <int FT>
__global__ __launch_bounds__(256) void binary_mul_kernel(void* __restrict__ y, const void* __restrict__ a,
                                                         const void* __restrict__ b, size_t count) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t)gridDim.x * 256)
    store_ft<FT>(y, i, load_ft<FT>(a, i) * load_ft<FT>(b, i));
}
template <int FT>
__global__ __launch_bounds__(256) void unary_kernel(void* __restrict__ y, const void* __restrict__ x, size_t count, int act) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t)gridDim.x * 256)
    store_ft<FT>(y, i, apply_act(load_ft<FT>(x, i), act));
}
// out[row, col] = f(in[row, col]) * in[row, inner + col]  (unary_glu_kernel, unary.cu:120-133; f's result rounded to FT first)
template <int FT>
__global__ __launch_bounds__(256) void unary_glu_kernel(void* __restrict__ y, const void* __restrict__ x, size_t outer, size_t inner,
                                                        int act) {
  const size_t count = outer * inner;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t)gridDim.x * 256) {
    const size_t row = i / inner, col = i - row * inner;
    float f = apply_act(load_ft<FT>(x, row * inner * 2 + col), act);
    if constexpr (FT != DIHIP_F32) f = ft_round<FT>(f);
    store_ft<FT>(y, i, f * load_ft<FT>(x, row * inner * 2 + inner + col));
  }
}
// EmbeddingT5 with an FT output (embeddingT5.cu): out[m, :] = table[clamp(ids[m]), :]
template <int FT>
__global__ __launch_bounds__(256) void embedding_ft_kernel(void* __restrict__ out, const int64_t* __restrict__ ids,
                                                           const void* __restrict__ table, int K, int vocab) {
  const int m = blockIdx.x;
  int64_t id = ids[m];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const size_t row = (size_t)id * K;
  for (int k = threadIdx.x; k < K; k += 256) store_ft<FT>(out, (size_t)m * K + k, load_ft<FT>(table, row + k));
}
template <int FT>
__global__ __launch_bounds__(256) void cast_to_f32_kernel(float* __restrict__ y, const void* __restrict__ x, size_t count) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t)gridDim.x * 256) y[i] = load_ft<FT>(x, i);
}

// ---- greedy argmax (GenerateOp top_k = 1): lowest index wins ties --------------------------------
struct ArgPair {
  float v;
  int i;
};
// NAN_FIRST: a NaN before any number, as torch.argmax has it (else it is passed over)
template <bool NAN_FIRST = false>
__device__ __forceinline__ ArgPair arg_better(ArgPair a, ArgPair b) {
  if constexpr (NAN_FIRST) {
    const bool an = a.v != a.v, bn = b.v != b.v;
    if (an || bn) return bn && (!an || b.i < a.i) ? b : a;
  }
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
template <bool NAN_FIRST = false>
__device__ __forceinline__ ArgPair wave_argmax(ArgPair p) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgPair q{__shfl_xor(p.v, o, 64), __shfl_xor(p.i, o, 64)};
    p = arg_better<NAN_FIRST>(p, q);
  }
  return p;
}
// stage 1: grid (blocks, M) -> partial[m][block]; stage 2: one wave per row.  Bound by launch and latency: four neighbours per load and four loads in flight where rows come in
// 16-byte pieces (152064 columns, one row: 5.6 -> 4.7 us, 32 rows 6.7 -> 5.8)
template <bool NAN_FIRST>
__global__ __launch_bounds__(256) void argmax_stage1(ArgPair* __restrict__ partial, const float* __restrict__ logits,
                                                     int N) {
  __shared__ ArgPair red[4];
  const int m = blockIdx.y;
  ArgPair best{-INFINITY, 0x7fffffff};
  const float* row = logits + (size_t)m * N;
  if (N % 4 == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0) {   // (uniform)
    const int quads = N / 4, step = gridDim.x * 256;
    for (int q = blockIdx.x * 256 + threadIdx.x; q < quads; q += 4 * step) {
      f32x4_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const f32x4_t*>(row + (size_t)min(q + u * step, quads - 1) * 4);   // (past the end: the last again)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) best = arg_better<NAN_FIRST>(best, ArgPair{v[u][r], min(q + u * step, quads - 1) * 4 + r});
    }
  } else {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < N; i += gridDim.x * 256) best = arg_better<NAN_FIRST>(best, ArgPair{row[i], i});
  }
  best = wave_argmax<NAN_FIRST>(best);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    ArgPair r = arg_better<NAN_FIRST>(arg_better<NAN_FIRST>(red[0], red[1]), arg_better<NAN_FIRST>(red[2], red[3]));
    partial[(size_t)m * gridDim.x + blockIdx.x] = r;
  }
}
// adv_a / adv_b (optional): per-request u32 counters (sequence lengths) advanced by one with the sampled id
template <bool NAN_FIRST>
__global__ __launch_bounds__(64) void argmax_stage2(int64_t* __restrict__ ids, const ArgPair* __restrict__ partial,
                                                    int nblocks, uint32_t* adv_a, uint32_t* adv_b) {
  const int m = blockIdx.x;
  ArgPair r{-INFINITY, 0x7fffffff};
  for (int i = threadIdx.x; i < nblocks; i += 64) r = arg_better<NAN_FIRST>(r, partial[(size_t)m * nblocks + i]);
  r = wave_argmax<NAN_FIRST>(r);
  if (threadIdx.x == 0) {
    ids[m] = r.i == 0x7fffffff ? 0 : (int64_t)r.i;  // an all-NaN row never beats the sentinel: a valid id, not 2^31 - 1
    if (adv_a) adv_a[m] += 1u;
    if (adv_b) adv_b[m] += 1u;
  }
}

// one wave per row: best of `count` pairs at in[m*row_stride + i*elem_stride]; writes the id and/or
// the pair (index shifted by index_offset)
__global__ __launch_bounds__(64) void argmax_merge_kernel(int64_t* ids, ArgPair* pairs_out, const ArgPair* in, int count,
                                                          int row_stride, int elem_stride, int index_offset) {
  const int m = blockIdx.x;
  ArgPair best{-INFINITY, 0x7fffffff};
  for (int i = threadIdx.x; i < count; i += 64) best = arg_better(best, in[(size_t)m * row_stride + (size_t)i * elem_stride]);
  best = wave_argmax(best);
  if (threadIdx.x == 0) {
    if (ids) ids[m] = best.i == 0x7fffffff ? 0 : (int64_t)best.i;
    if (pairs_out) pairs_out[m] = ArgPair{best.v, best.i == 0x7fffffff ? best.i : best.i + index_offset};  // sentinel stays a sentinel
  }
}

template <int FT>
__global__ __launch_bounds__(256) void embedding_kernel(float* __restrict__ h, const int64_t* __restrict__ ids,
                                                        const void* __restrict__ table, int K, int vocab) {
  const int m = blockIdx.x;
  int64_t id = ids[m];
  if (vocab > 0) id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);  // an id out of range reads a valid row instead of faulting
  const size_t row = (size_t)id * K;
  const int k_lo = blockIdx.y * 1024, k_hi = min(K, k_lo + 1024);   // (a row over several workgroups: one of 3584 5.8 -> 4.7 us, 32 8.3 -> 4.7)
#pragma unroll 4
  for (int k = k_lo + threadIdx.x; k < k_hi; k += 256) h[(size_t)m * K + k] = load_ft<FT>(table, row + k);
}

// the state of a decoding step as a caller gives it: next tokens, tokens in the cache, the same with the one to come.  Three copies and an addition otherwise (14.5 + 4.9 us
// of kernels and the gaps between them -> 4.8)
__global__ __launch_bounds__(64) void decode_state_kernel(int64_t* ids, uint32_t* old_lens, uint32_t* new_lens, const int64_t* ids_in, const int32_t* lens_in, int B) {
  const int b = blockIdx.x * 64 + threadIdx.x;
  if (b >= B) return;
  const int64_t id = ids_in[b];
  const uint32_t len = (uint32_t)lens_in[b];
  ids[b] = id;
  old_lens[b] = len;
  new_lens[b] = len + 1u;
}

__global__ void increment_u32_kernel(uint32_t* v, int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) v[i] += 1u;
}

constexpr int ARGMAX_BLOCKS = 64;

}  // namespace dihip

using namespace dihip;

#define FT_SWITCH(dtype, BODY)                                         \
  switch (dtype) {                                                     \
    case DIHIP_F32: { constexpr int FT = DIHIP_F32; BODY; } break;     \
    case DIHIP_F16: { constexpr int FT = DIHIP_F16; BODY; } break;     \
    case DIHIP_BF16: { constexpr int FT = DIHIP_BF16; BODY; } break;   \
    default:                                                           \
      set_last_error("unsupported dtype %d", dtype);                   \
      return DIHIP_PARAM_ERROR;                                        \
  }

// Weight prefetch into the 256 MB Infinity Cache (memory-side): streams up to 8 buffers through the
// load path and discards them.  Launched on a SIDE stream next to a latency-bound phase of the decode
// step (attention at batch 1 leaves HBM idle), so that the following weight-streaming GEMVs find their
// weights on-die.  Reads only; the never-true store keeps the loads alive.
struct PrefetchArgs {
  const u32x4_t* p[8];
  size_t n16[8];  // 16-byte vectors per buffer
  unsigned* sink;
};
__global__ __launch_bounds__(256) void prefetch_kernel(const PrefetchArgs a) {
  unsigned acc = 0;
  const size_t stride = (size_t)gridDim.x * 256;
  for (int b = 0; b < 8; ++b) {
    const u32x4_t* p = a.p[b];
    const size_t n = a.n16[b];
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (; i + 7 * stride < n; i += 8 * stride) {
      u32x4_t v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = p[i + j * stride];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc ^= v[j][0] ^ v[j][3];
    }
    for (; i < n; i += stride) acc ^= p[i][0];
  }
  if (acc == 0x9E3779B9u && a.sink) a.sink[0] = acc;  // practically never
}

extern "C" {

int dihip_rmsnorm(void* stream, void* y, const void* x, const void* gamma, float eps, int rows, int cols, int dtype) {
  DIHIP_REQUIRE(rows >= 0 && cols > 0 && y && x && gamma, DIHIP_PARAM_ERROR, "rmsnorm: bad argument");
  if (rows == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  FT_SWITCH(dtype, hipLaunchKernelGGL((rmsnorm_kernel<FT>), dim3(rows), dim3(256), 0, s, y, x, gamma, eps, cols));
  return launch_status();
}

int dihip_rope_qk(void* stream, void* qkv, const uint32_t* positions, const float* inv_freq, int rows, int num_heads,
                  int num_groups, int head_size, int dtype) {
  DIHIP_REQUIRE(rows >= 0 && num_heads > 0 && num_groups > 0 && qkv && positions && inv_freq, DIHIP_PARAM_ERROR,
                "rope: bad argument");
  DIHIP_REQUIRE(head_size > 0 && head_size <= 128 && head_size % 2 == 0, DIHIP_PARAM_ERROR, "rope: head size %d",
                head_size);
  if (rows == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  FT_SWITCH(dtype, hipLaunchKernelGGL((rope_qk_kernel<FT>), dim3(rows, num_heads + num_groups), dim3(64), 0, s, qkv,
                                      positions, inv_freq, num_heads, num_groups, head_size));
  return launch_status();
}

int dihip_binary_add(void* stream, void* y, const void* a, const void* b, size_t count, int dtype) {
  DIHIP_REQUIRE(y && a && b, DIHIP_PARAM_ERROR, "binary_add: null pointer");
  if (count == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (int)std::min<size_t>((count + 255) / 256, 2048);
  FT_SWITCH(dtype, hipLaunchKernelGGL((binary_kernel<FT, 0>), dim3(blocks), dim3(256), 0, s, y, a, b, count));
  return launch_status();
}

int dihip_silu_mul(void* stream, void* y, const void* gate, const void* up, size_t count, int dtype) {
  DIHIP_REQUIRE(y && gate && up, DIHIP_PARAM_ERROR, "silu_mul: null pointer");
  if (count == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (int)std::min<size_t>((count + 255) / 256, 2048);
  FT_SWITCH(dtype, hipLaunchKernelGGL((binary_kernel<FT, 1>), dim3(blocks), dim3(256), 0, s, y, gate, up, count));
  return launch_status();
}

int dihip_binary_mul(void* stream, void* y, const void* a, const void* b, size_t count, int dtype) {
  DIHIP_REQUIRE(y && a && b, DIHIP_PARAM_ERROR, "binary_mul: null pointer");
  if (count == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (int)std::min<size_t>((count + 255) / 256, 2048);
  FT_SWITCH(dtype, hipLaunchKernelGGL((binary_mul_kernel<FT>), dim3(blocks), dim3(256), 0, s, y, a, b, count));
  return launch_status();
}

int dihip_unary(void* stream, void* y, const void* x, size_t count, int act, int dtype) {
  DIHIP_REQUIRE(y && x, DIHIP_PARAM_ERROR, "unary: null pointer");
  DIHIP_REQUIRE(act >= DIHIP_ACT_NONE && act <= DIHIP_ACT_SIGMOID, DIHIP_PARAM_ERROR, "unary: unknown UnaryType %d", act);
  if (count == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (int)std::min<size_t>((count + 255) / 256, 2048);
  FT_SWITCH(dtype, hipLaunchKernelGGL((unary_kernel<FT>), dim3(blocks), dim3(256), 0, s, y, x, count, act));
  return launch_status();
}

int dihip_unary_glu(void* stream, void* y, const void* x, size_t outer, size_t inner, int act, int dtype) {
  DIHIP_REQUIRE(y && x, DIHIP_PARAM_ERROR, "unary_glu: null pointer");
  DIHIP_REQUIRE(act >= DIHIP_ACT_NONE && act <= DIHIP_ACT_SIGMOID, DIHIP_PARAM_ERROR, "unary_glu: unknown UnaryType %d", act);
  if (outer * inner == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (int)std::min<size_t>((outer * inner + 255) / 256, 2048);
  FT_SWITCH(dtype, hipLaunchKernelGGL((unary_glu_kernel<FT>), dim3(blocks), dim3(256), 0, s, y, x, outer, inner, act));
  return launch_status();
}

int dihip_embedding_ft(void* stream, void* out, const int64_t* ids, const void* table, int M, int K, int vocab, int dtype) {
  DIHIP_REQUIRE(M >= 0 && K > 0 && vocab > 0 && out && ids && table, DIHIP_PARAM_ERROR, "embedding_ft: bad argument");
  if (M == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  FT_SWITCH(dtype, hipLaunchKernelGGL((embedding_ft_kernel<FT>), dim3(M), dim3(256), 0, s, out, ids, table, K, vocab));
  return launch_status();
}

int dihip_cast_to_f32(void* stream, float* y, const void* x, size_t count, int dtype) {
  DIHIP_REQUIRE(y && x, DIHIP_PARAM_ERROR, "cast_to_f32: null pointer");
  if (count == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int blocks = (int)std::min<size_t>((count + 255) / 256, 2048);
  FT_SWITCH(dtype, hipLaunchKernelGGL((cast_to_f32_kernel<FT>), dim3(blocks), dim3(256), 0, s, y, x, count));
  return launch_status();
}

}  // extern "C"
template <bool NAN_FIRST>
static int argmax_launch(const char* what, void* stream, int64_t* ids, const float* logits, int M, int N, void* ws, size_t ws_bytes, uint32_t* counters_a, uint32_t* counters_b) {
  DIHIP_REQUIRE(M >= 0 && N > 0 && ids && logits, DIHIP_PARAM_ERROR, "%s: bad argument", what);
  if (M == 0) return DIHIP_SUCCESS;
  DIHIP_REQUIRE(ws && ws_bytes >= (size_t)M * ARGMAX_BLOCKS * sizeof(ArgPair), DIHIP_MEMORY_ERROR,
                "%s: workspace needs %zu bytes", what, (size_t)M * ARGMAX_BLOCKS * sizeof(ArgPair));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(argmax_stage1<NAN_FIRST>, dim3(ARGMAX_BLOCKS, M), dim3(256), 0, s, (ArgPair*)ws, logits, N);
  hipLaunchKernelGGL(argmax_stage2<NAN_FIRST>, dim3(M), dim3(64), 0, s, ids, (const ArgPair*)ws, ARGMAX_BLOCKS, counters_a, counters_b);
  return launch_status();
}
extern "C" {

int dihip_argmax(void* stream, int64_t* ids, const float* logits, int M, int N, void* ws, size_t ws_bytes) {
  return argmax_launch<false>("argmax", stream, ids, logits, M, N, ws, ws_bytes, nullptr, nullptr);
}

int dihip_argmax_nan_first(void* stream, int64_t* ids, const float* logits, int M, int N, void* ws, size_t ws_bytes) {
  return argmax_launch<true>("argmax_nan_first", stream, ids, logits, M, N, ws, ws_bytes, nullptr, nullptr);
}

int dihip_argmax_advance(void* stream, int64_t* ids, const float* logits, int M, int N, void* ws, size_t ws_bytes,
                         uint32_t* counters_a, uint32_t* counters_b) {
  return argmax_launch<false>("argmax_advance", stream, ids, logits, M, N, ws, ws_bytes, counters_a, counters_b);
}

// TP vocabulary-parallel greedy sampling: each rank reduces its logits slice to one (value, global
// index) pair per row, the pairs are all-gathered, and every rank merges them identically.
int dihip_argmax_partial(void* stream, void* pairs_out, const float* logits, int M, int N, int index_offset, void* ws,
                         size_t ws_bytes) {
  DIHIP_REQUIRE(M >= 0 && N > 0 && pairs_out && logits, DIHIP_PARAM_ERROR, "argmax_partial: bad argument");
  if (M == 0) return DIHIP_SUCCESS;
  DIHIP_REQUIRE(ws && ws_bytes >= (size_t)M * ARGMAX_BLOCKS * sizeof(ArgPair), DIHIP_MEMORY_ERROR,
                "argmax_partial: workspace needs %zu bytes", (size_t)M * ARGMAX_BLOCKS * sizeof(ArgPair));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(argmax_stage1<false>, dim3(ARGMAX_BLOCKS, M), dim3(256), 0, s, (ArgPair*)ws, logits, N);
  hipLaunchKernelGGL(argmax_merge_kernel, dim3(M), dim3(64), 0, s, (int64_t*)nullptr, (ArgPair*)pairs_out,
                     (const ArgPair*)ws, ARGMAX_BLOCKS, ARGMAX_BLOCKS, 1, index_offset);
  return launch_status();
}

int dihip_argmax_merge(void* stream, int64_t* ids, const void* pairs, int nparts, int M) {
  DIHIP_REQUIRE(M >= 0 && nparts > 0 && ids && pairs, DIHIP_PARAM_ERROR, "argmax_merge: bad argument");
  if (M == 0) return DIHIP_SUCCESS;
  // pairs laid out [nparts][M] (all-gather order)
  hipLaunchKernelGGL(argmax_merge_kernel, dim3(M), dim3(64), 0, reinterpret_cast<hipStream_t>(stream), ids,
                     (ArgPair*)nullptr, (const ArgPair*)pairs, nparts, 1, M, 0);
  return launch_status();
}

int dihip_embedding(void* stream, float* h, const int64_t* ids, const void* table, int M, int K, int dtype) {
  DIHIP_REQUIRE(M >= 0 && K > 0 && h && ids && table, DIHIP_PARAM_ERROR, "embedding: bad argument");
  if (M == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  FT_SWITCH(dtype, hipLaunchKernelGGL((embedding_kernel<FT>), dim3(M, (K + 1023) / 1024), dim3(256), 0, s, h, ids, table, K, 0));
  return launch_status();
}

int dihip_embedding_v(void* stream, float* h, const int64_t* ids, const void* table, int M, int K, int vocab, int dtype) {
  DIHIP_REQUIRE(M >= 0 && K > 0 && vocab > 0 && h && ids && table, DIHIP_PARAM_ERROR, "embedding: bad argument");
  if (M == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  FT_SWITCH(dtype, hipLaunchKernelGGL((embedding_kernel<FT>), dim3(M, (K + 1023) / 1024), dim3(256), 0, s, h, ids, table, K, vocab));
  return launch_status();
}

int dihip_decode_state(void* stream, int64_t* ids, uint32_t* old_lens, uint32_t* new_lens, const int64_t* ids_in, const int32_t* lens_in, int B) {
  DIHIP_REQUIRE(B >= 0 && ids && old_lens && new_lens && ids_in && lens_in, DIHIP_PARAM_ERROR, "decode_state: bad argument");
  if (B == 0) return DIHIP_SUCCESS;
  hipLaunchKernelGGL(decode_state_kernel, dim3((B + 63) / 64), dim3(64), 0, reinterpret_cast<hipStream_t>(stream), ids, old_lens, new_lens, ids_in, lens_in, B);
  return launch_status();
}

int dihip_increment_u32(void* stream, uint32_t* v, int count) {
  DIHIP_REQUIRE(count >= 0 && v, DIHIP_PARAM_ERROR, "increment: bad argument");
  if (count == 0) return DIHIP_SUCCESS;
  hipLaunchKernelGGL(increment_u32_kernel, dim3((count + 255) / 256), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), v, count);
  return launch_status();
}

int dihip_prefetch(void* stream, const void* const* bufs, const size_t* bytes, int count, int num_workgroups) {
  DIHIP_REQUIRE(count >= 0 && count <= 8 && (count == 0 || (bufs && bytes)), DIHIP_PARAM_ERROR, "prefetch: bad argument");
  if (count == 0) return DIHIP_SUCCESS;
  PrefetchArgs a{};
  for (int i = 0; i < count; ++i) {
    DIHIP_REQUIRE((reinterpret_cast<uintptr_t>(bufs[i]) & 15) == 0, DIHIP_PARAM_ERROR, "prefetch: buffers must be 16-byte aligned");
    a.p[i] = reinterpret_cast<const u32x4_t*>(bufs[i]);
    a.n16[i] = bytes[i] / 16;
  }
  a.sink = nullptr;
  if (num_workgroups <= 0) num_workgroups = 256;
  hipLaunchKernelGGL(prefetch_kernel, dim3(num_workgroups), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), a);
  return launch_status();
}

}  // extern "C"
