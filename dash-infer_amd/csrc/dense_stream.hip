// dense_stream.hip -- the output matrix of a language model for 5 .. 32 rows: logits f32 [M, N] = x . W, W 16-bit in tile-major order
// ([16-column tile][32 of K][lane][16 bytes]), x in the FRAG32 layout (device_utils.h).
//
// Bound by the weights' bytes (152064 x 3584: 1.09 GB).  The general kernel re-reads the rows for every few column tiles and keeps its loads
// short; here one workgroup per CU lives for the whole launch:
//   * it owns up to 40 neighbouring column tiles, 8 waves take them in turn and keep ALL their accumulators (5 tiles x 8 registers at 32 rows);
//   * the rows' operands lie in LDS -- all of K where they fit (16 rows x 3584), else one range of K after the other, each for all tiles --: they
//     are read from the L2 once per CU, and the walk itself issues nothing but weight loads;
//   * a wave asks for the next 8 KiB (the next batch of its tile, of its next tile, of the next range) before it multiplies the present ones: the
//     stream does not stop at the ends of tiles.
// 32 / 16 / 7 rows of 152064 x 3584: 210 / 198 / 196 us (the general kernel) -> 182 / 182 / 177 (6.0 - 6.2 TB/s).  What is left: 37 tiles are not 8 waves'
// equal shares (the last fifth of the time runs on five waves), and the rows' way into LDS before the stream.
#include "gemm_lowp_kernel.hpp"  // mfma16<FT>

namespace dihip {
namespace {

constexpr int DS_WAVES = 8, DS_TILES = 5, DS_U = 8;   // column tiles per wave, K steps (of 32) per batch

template <int FT, int MT>
__global__ __launch_bounds__(64 * DS_WAVES, 2) void dense_stream_kernel(const u32x4_t* __restrict__ w, const u32x4_t* __restrict__ x, float* __restrict__ out,
                                                                        int M, int N, int KT, int ntiles, int range) {
  extern __shared__ __attribute__((aligned(16))) u32x4_t xs[];   // [K step of the range][MT][64]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = (int)((long)ntiles * blockIdx.x / gridDim.x), hi = (int)((long)ntiles * (blockIdx.x + 1) / gridDim.x);
  const int mine = max(0, (hi - lo - wave + DS_WAVES - 1) / DS_WAVES);   // tiles lo + wave + 8 i
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[DS_TILES][MT];
#pragma unroll
  for (int i = 0; i < DS_TILES; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[i][m] = z4;
  auto load = [&](u32x4_t (&d)[DS_U], const u32x4_t* p) {
#pragma unroll
    for (int u = 0; u < DS_U; ++u) d[u] = __builtin_nontemporal_load(p + u * 64);
  };
  auto mul = [&](u32x4_t (&d)[DS_U], int b, f32x4_t (&c)[MT]) {
#pragma unroll
    for (int u = 0; u < DS_U; ++u)
#pragma unroll
      for (int m = 0; m < MT; ++m) c[m] = mfma16<FT>(d[u], xs[((b + u) * MT + m) * 64 + lane], c[m]);
  };
  auto tile = [&](int i) { return w + (size_t)(lo + wave + DS_WAVES * i) * KT * 64 + lane; };
  u32x4_t wa[DS_U], wb[DS_U];     // two batches in turn
  if (mine > 0) load(wa, tile(0));
  for (int k0 = 0; k0 < KT; k0 += range) {
    const int kn = min(range, KT - k0);
    if (k0) __syncthreads();                    // the range before has been read
    for (int e = tid; e < kn * MT * 64; e += 64 * DS_WAVES) xs[e] = x[(size_t)k0 * MT * 64 + e];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DS_TILES; ++i) {
      if (i < mine) {                           // (uniform)
        const u32x4_t* p = tile(i) + (size_t)k0 * 64;
        // what follows the tile: the next one, the first one's next range, or (the walk's end) this batch once more
        const u32x4_t* then = i + 1 < mine ? tile(i + 1) + (size_t)k0 * 64 : k0 + range < KT ? tile(0) + (size_t)(k0 + range) * 64 : p;
        for (int b = 0; b < kn; b += 2 * DS_U) {
          load(wb, p + DS_U * 64);
          __builtin_amdgcn_sched_barrier(0);
          mul(wa, b, acc[i]);
          p = b + 2 * DS_U < kn ? p + 2 * DS_U * 64 : then;
          load(wa, p);
          __builtin_amdgcn_sched_barrier(0);
          mul(wb, b + DS_U, acc[i]);
        }
      }
    }
  }
  // the weights were the A operand: a lane holds 4 neighbouring columns of row m * 16 + lane % 16
#pragma unroll
  for (int i = 0; i < DS_TILES; ++i) {
    if (i < mine) {
      const int n = (lo + wave + DS_WAVES * i) * 16 + (lane >> 4) * 4;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = m * 16 + (lane & 15);
        if (row < M) {
          if (n + 3 < N && N % 4 == 0) {
            *reinterpret_cast<f32x4_t*>(out + (size_t)row * N + n) = acc[i][m];
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < N) out[(size_t)row * N + n + r] = acc[i][m][r];
          }
        }
      }
    }
  }
}

template <int FT, int MT>
int go(hipStream_t s, const void* w, const void* x, float* out, int M, int N, int KT, int ntiles) {
  constexpr int LDS_STEPS = 152 / MT / (2 * DS_U) * (2 * DS_U);          // K steps of the rows' operands in 152 KiB, in whole pairs of batches
  const int ranges = (KT + LDS_STEPS - 1) / LDS_STEPS, range = ((KT + ranges - 1) / ranges + 2 * DS_U - 1) / (2 * DS_U) * (2 * DS_U);
  const size_t lds = (size_t)std::min(range, KT) * MT * 1024;
  auto kern = dense_stream_kernel<FT, MT>;
  DIHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), DIHIP_RUNTIME_ERROR);
  int ncu = cached_num_cus();
  if (ncu <= 0) ncu = 256;
  const int most = DS_WAVES * DS_TILES;        // tiles of a workgroup
  const int rounds = (ntiles + ncu * most - 1) / (ncu * most);
  hipLaunchKernelGGL(kern, dim3(ncu * rounds), dim3(64 * DS_WAVES), lds, s, (const u32x4_t*)w, (const u32x4_t*)x, out, M, N, KT, ntiles, range);
  return launch_status();
}

}  // namespace

// 5 .. 32 rows, K in whole pairs of batches, at least four column tiles per CU (below, too few waves have a tile)
bool dense_stream_takes(int M, int N, int K) {
  int ncu = cached_num_cus();
  if (ncu <= 0) ncu = 256;
  return M > 4 && M <= 32 && K % (2 * DS_U * 32) == 0 && K > 0 && (N + 15) / 16 >= 4 * ncu;
}

int launch_dense_stream(hipStream_t s, const void* w, const void* x_frag, float* out, int M, int N, int K, int dtype) {
  const int KT = K / 32, ntiles = (N + 15) / 16;
  DIHIP_REQUIRE(reinterpret_cast<uintptr_t>(out) % 16 == 0 || N % 4 != 0, DIHIP_PARAM_ERROR, "lm_head: the logits must be 16-byte aligned");
  if (dtype == DIHIP_F16) return M <= 16 ? go<DIHIP_F16, 1>(s, w, x_frag, out, M, N, KT, ntiles) : go<DIHIP_F16, 2>(s, w, x_frag, out, M, N, KT, ntiles);
  return M <= 16 ? go<DIHIP_BF16, 1>(s, w, x_frag, out, M, N, KT, ntiles) : go<DIHIP_BF16, 2>(s, w, x_frag, out, M, N, KT, ntiles);
}

}  // namespace dihip
