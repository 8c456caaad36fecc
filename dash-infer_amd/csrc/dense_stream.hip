// dense_stream.hip -- the output matrix of a language model for 5 .. 32 rows: logits f32 [M, N] = x . W, W 16-bit in tile-major order
// ([16-column tile][32 of K][lane][16 bytes]), x in the FRAG32 layout (device_utils.h).
//
// Bound by the weights' bytes (152064 x 3584: 1.09 GB).  The general kernel re-reads the rows for every few column tiles and keeps its loads
// short; here one workgroup per CU lives for the whole launch:
//   * it owns up to 40 neighbouring column tiles; each of its 8 waves walks an eighth of them, counted in batches of 16 steps of K -- 37 tiles are not 8 waves' equal shares,
//     and a wave is bound by its own loads' way: with whole tiles (five or four a wave) the last fifth of the time ran on five waves.  It keeps all its accumulators (6 tiles x 8
//     registers at 32 rows); the sums of a tile that two waves share meet in LDS at the end;
//   * the rows' operands lie in LDS -- all of K where they fit (16 rows x 3584), else one range of K after the other, each for all tiles --: they
//     are read from the L2 once per CU, and the walk itself issues nothing but weight loads;
//   * a wave asks for the next 8 KiB (the next batch of its tile, of its next tile, of the next range) before it multiplies the present ones: the
//     stream does not stop at the ends of tiles.
// 32 / 16 / 7 rows of 152064 x 3584: 210 / 198 / 196 us (the general kernel) -> 182 / 182 / 177 (whole tiles) -> 176 / 174 / 173 (even shares: 6.2 TB/s).  What is left: the rows' way into LDS before the
// stream (and between the ranges of K).
#include "gemm_lowp_kernel.hpp"  // mfma16<FT>

namespace dihip {
namespace {

constexpr int DS_WAVES = 8, DS_TILES = 5, DS_SLOTS = DS_TILES + 1, DS_U = 8;   // column tiles per wave, tiles it may touch, K steps (of 32) per batch of loads
constexpr int DS_UNIT = 2 * DS_U;   // K steps: what the waves' shares are counted in

template <int FT, int MT>
__global__ __launch_bounds__(64 * DS_WAVES, 2) void dense_stream_kernel(const u32x4_t* __restrict__ w, const u32x4_t* __restrict__ x, float* __restrict__ out,
                                                                        int M, int N, int KT, int ntiles, int range) {
  extern __shared__ __attribute__((aligned(16))) u32x4_t xs[];   // [K step of the range][MT][64]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = (int)((long)ntiles * blockIdx.x / gridDim.x), hi = (int)((long)ntiles * (blockIdx.x + 1) / gridDim.x);
  // wave w's share of T tiles begins T w / 8 tiles in: tiles first .. first + 5; in every range of K it is [T upt w / 8, T upt (w + 1) / 8) of the range's units (upt: units per
  // tile), which lie in the same tiles whatever upt is
  const int T = hi - lo, first = T * wave / DS_WAVES;
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[DS_SLOTS][MT];
#pragma unroll
  for (int i = 0; i < DS_SLOTS; ++i)
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
  auto tile = [&](int i) { return w + (size_t)(lo + first + i) * KT * 64 + lane; };
  auto begin = [&](int wv, int upt) { return T * upt * wv / DS_WAVES; };
  // the wave's first batch of the ranges from k0 on; it has none: its first tile's (loaded, not used)
  auto start = [&](int k0) {
    for (; k0 < KT; k0 += range) {
      const int upt = min(range, KT - k0) / DS_UNIT, u = begin(wave, upt);
      if (u < begin(wave + 1, upt)) return tile(0) + (size_t)(k0 + (u - first * upt) * DS_UNIT) * 64;
    }
    return w + (size_t)min(lo + first, ntiles - 1) * KT * 64 + lane;
  };
  u32x4_t wa[DS_U], wb[DS_U];     // two batches in turn
  load(wa, start(0));
  for (int k0 = 0; k0 < KT; k0 += range) {
    const int kn = min(range, KT - k0), upt = kn / DS_UNIT, u0 = begin(wave, upt), u1 = begin(wave + 1, upt);
    if (k0) __syncthreads();                    // the range before has been read
    constexpr int AHEAD = 10;                   // (a thread's loads in flight: all of a range in two goes)
    const u32x4_t* const from = x + (size_t)k0 * MT * 64;
    for (int e = tid; e < kn * MT * 64; e += AHEAD * 64 * DS_WAVES) {
      u32x4_t r[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) r[j] = from[min(e + j * 64 * DS_WAVES, kn * MT * 64 - 1)];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j)
        if (e + j * 64 * DS_WAVES < kn * MT * 64) xs[e + j * 64 * DS_WAVES] = r[j];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DS_SLOTS; ++i) {
      const int at = (first + i) * upt, b0 = max(u0 - at, 0) * DS_UNIT, b1 = min(u1 - at, upt) * DS_UNIT;   // (uniform) this tile's part of the share
      if (b0 < b1) {
        const u32x4_t* p = tile(i) + (size_t)(k0 + b0) * 64;
        const u32x4_t* then = u1 > at + upt ? tile(i + 1) + (size_t)k0 * 64 : start(k0 + range);   // what follows: the next tile, or the next range
        for (int b = b0; b < b1; b += DS_UNIT) {
          load(wb, p + DS_U * 64);
          __builtin_amdgcn_sched_barrier(0);
          mul(wa, b, acc[i]);
          p = b + DS_UNIT < b1 ? p + DS_UNIT * 64 : then;
          load(wa, p);
          __builtin_amdgcn_sched_barrier(0);
          mul(wb, b + DS_U, acc[i]);
        }
      }
    }
  }
  // a share that begins inside a tile leaves its sums of it to the wave that has the tile's beginning, which adds them in the waves' order
  __syncthreads();
  f32x4_t* const part = reinterpret_cast<f32x4_t*>(xs);   // [wave][MT][64]
  if (T * wave % DS_WAVES != 0) {
#pragma unroll
    for (int m = 0; m < MT; ++m) part[(wave * MT + m) * 64 + lane] = acc[0][m];
  }
  __syncthreads();
  // the weights were the A operand: a lane holds 4 neighbouring columns of row m * 16 + lane % 16
#pragma unroll
  for (int i = 0; i < DS_SLOTS; ++i) {
    const int t = first + i;
    if (t < T && DS_WAVES * t < T * (wave + 1) && (i > 0 || T * wave % DS_WAVES == 0)) {   // (uniform) the tile's beginning is this wave's
      for (int o = wave + 1; o < DS_WAVES && T * o / DS_WAVES == t && T * o % DS_WAVES != 0; ++o) {
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[i][m] += part[(o * MT + m) * 64 + lane];
      }
      const int n = (lo + t) * 16 + (lane >> 4) * 4;
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
  const size_t lds = (size_t)std::max(std::min(range, KT), DS_WAVES) * MT * 1024;   // (the rows, at the end the shared tiles' sums)
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
