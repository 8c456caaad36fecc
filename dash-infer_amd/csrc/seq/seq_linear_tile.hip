// seq_linear_tile.hip -- linear_pipe_kernel: products of many bf16 rows (prompts, portions) with bf16 weights, on the matrix cores.
//
// A tile of 256 x 256 (8 waves, 128 x 64 each; smaller ones below) walks K in steps of 64 through two LDS slots:
//   * rows and weights go straight into LDS (global_load_lds, 16 bytes a lane): no registers and no instructions for staging.  A 1 KiB piece is 8
//     rows x 128 bytes in the order of the lanes (whole cache lines: with 64-byte pieces the L2s had twice the requests, 236 against
//     226 us), so the 16-byte chunks of a row change places on the memory side (chunk ^ row % 8) and the operand reads of 8
//     consecutive lanes touch every bank once;
//   * a step is two halves of 32.  While the first multiplies, the operands of the second are read; then one barrier tells that this slot has
//     been read and the next one has landed (its loads are a whole step old); while the second half multiplies, the slot is
//     refilled for the step after the next and the next step's first operands are read.  The tail re-reads the last step instead of
//     branching;
//   * the order of products, reads and loads is pinned (sched_barrier): left alone the compiler moves the reads behind the products;
//   * the loads are inline asm (they return nothing into registers): the compiler would count them into every wait for an LDS read.
// 2048 rows, 4096 -> 14336 (f32 out): 375 us (640 TFLOP/s, the register-staged kernel of seq_linear.hip) -> 220 us (1090); the matrix pipes are
// busy 50 % of the time at 2.0 GHz, the second round of 448 tiles on 256 CUs costs an eighth and the results' way out a tenth.
// A 128 x 128 tile (4 waves, two workgroups per CU) reads twice as much per product and serves what 256 x 256 tiles cut badly.
//
// Narrow outputs and short prompts have too few tiles for 256 CUs: K is then split over workgroups that leave f32 tiles in a slab,
// and linear_parts_kernel adds them in order (plan_linear_tile).
#include "seq_linear.h"

namespace dihip {
namespace {

constexpr int LT_BK = 64, LT_SLOTS = 2;

// workgroups go round the 8 XCDs: XCD x gets the tiles x * (total / 8) .., neighbours, so that one L2 holds few weights
__device__ __forceinline__ int xcd_tile(int b, int total) {
  const int per = total / 8, rest = total % 8, x = b % 8, i = b / 8;
  return x * per + min(x, rest) + i;
}

// Segments: workgroup b takes the b-th of the tiles that hold rows -- group by group, the row tiles of a group side by side (they share its weights) --, false: there are
// fewer.  A grid over the bound on a segment's rows is mostly workgroups without rows, and each waits for 64 KB of LDS to find that out: 32 segments of about 16
// rows at a bound of 130, 4096 -> 4096, 316 us with them (bound 100, one row tile: 255).
__device__ __forceinline__ bool seg_tile(const int32_t* __restrict__ seg, int groups, int bm, int ntiles, int b, int& g, int& mt, int& nt) {
  const int lane = threadIdx.x & 63;
  auto scan = [&](int i0, int& mine) {   // row tiles of group i0 + lane; -> of the groups i0 .. up to it
    const int i = i0 + lane;
    mine = i < groups ? (max(seg[i + 1] - seg[i], 0) + bm - 1) / bm : 0;
    int upto = mine;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const int other = __shfl_up(upto, d, 64);
      if (lane >= d) upto += other;
    }
    return upto;
  };
  int mine, total = 0;
  for (int i0 = 0; i0 < groups; i0 += 64) total += __builtin_amdgcn_readlane(scan(i0, mine), 63);
  total *= ntiles;
  if (b >= total) return false;
  b = xcd_tile(b, total);
  int before = 0;
  for (int i0 = 0; i0 < groups; i0 += 64) {
    const int upto = scan(i0, mine);
    const uint64_t past = __builtin_amdgcn_ballot_w64((before + upto) * ntiles > b);
    if (past) {
      const int l = __builtin_ctzll(past), tiles = __builtin_amdgcn_readlane(mine, l), local = b - (before + __builtin_amdgcn_readlane(upto, l) - tiles) * ntiles;
      g = i0 + l;
      mt = local % tiles;
      nt = local / tiles;
      return true;
    }
    before += __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// MF / NF: 16-row operands of a wave along the rows (x) and the output columns (weight rows); WM x WN waves
// MAP: the rows of x are named by a map and may lie anywhere: 64-bit addresses per lane.  Else a tile's rows are neighbours: 32-bit offsets from its first
// GATED: half of a tile's columns are w's, half the same ones of w2 -- of every wave, so that both sums of an element meet in its piece of LDS.  What two launches
// cost beside the products: f32 sums out and in again, and the last round of tiles twice.  2048 rows 4096 -> 14336 twice 491 -> 444 us, 1500 rows 423 -> 334; 2048 -> 8192
// twice, 513 rows 92.7 -> 58.2, 128 rows 44.8 -> 28.7.
template <int MF, int NF, int WM, int WN, bool MAP, bool GATED>
__global__ __launch_bounds__(64 * WM * WN, (WM * WN) / 4) void linear_pipe_kernel(LinArgs a, int mtiles, int ntiles, int groups, bool vec4, int parts, float* slab) {
  constexpr int WAVES = WM * WN, BM = 16 * MF * WM, BN = 16 * NF * WN;
  constexpr int PIECES = (BM + BN) / 8, PER = PIECES / WAVES;     // 1 KiB pieces (8 rows x 128 bytes) of a K step, per wave
  static_assert(PIECES % WAVES == 0, "whole pieces per wave");
  constexpr int SLOT = PIECES * 1024;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int g = blockIdx.y, mt, nt;   // (the parts of a tile are blockIdx.z)
  if (a.seg) {
    if (!seg_tile(a.seg, groups, BM, ntiles, blockIdx.x, g, mt, nt)) return;
  } else {
    const int tile = xcd_tile(blockIdx.x, mtiles * ntiles);
    mt = tile % mtiles;
    nt = tile / mtiles;
  }
  int t_lo, t_hi;
  lin_rows(a, g, t_lo, t_hi);
  constexpr int HALVES = GATED ? 2 : 1, WCOLS = 16 * NF / HALVES;   // columns of y of a wave
  const int m0 = t_lo + mt * BM, n0 = nt * (BN / HALVES);
  if (m0 >= t_hi) return;
  const size_t xoff = (size_t)(g % a.xgroups) * a.xg;
  // pieces: first the rows of x, then those of w; lane l of a piece brings row l / 8, 16 bytes (l % 8) ^ (row % 8) of its 128
  const int prow = lane >> 3, pchunk = (lane & 7) ^ prow;
  const int all = a.K / LT_BK, part = blockIdx.z, k0 = (int)((long)all * part / parts), steps = (int)((long)all * (part + 1) / parts) - k0;
  const char* xbase = (const char*)((const uint16_t*)a.x + (MAP ? 0 : (size_t)m0 * a.ldx) + xoff + k0 * LT_BK);
  const char* wbase = (const char*)((const uint16_t*)a.w + ((size_t)g * a.N + n0) * a.K + k0 * LT_BK);
  const char* w2base = GATED ? (const char*)((const uint16_t*)a.w2 + (size_t)n0 * a.K + k0 * LT_BK) : nullptr;
  const char* base[PER];
  uint32_t off[PER];   // (the host checks that 256 rows lie within 2 GB)
  const char* addr[PER];   // (MAP, instead of both)
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int piece = wave * PER + p;
    const bool isx = piece < BM / 8;   // (uniform)
    int wrow = (piece - BM / 8) * 8;
    base[p] = isx ? xbase : wbase;
    if constexpr (GATED) {
      if (!isx && wrow % (2 * WCOLS) >= WCOLS) base[p] = w2base;
      wrow = wrow / (2 * WCOLS) * WCOLS + wrow % WCOLS;
    }
    const int r = isx ? min(m0 + piece * 8 + prow, t_hi - 1) : min(wrow + prow, a.N - 1 - n0);
    const size_t row = isx ? (MAP ? a.row_map[r] : r - m0) : r, from = (row * (size_t)(isx ? a.ldx : (long)a.K) + pchunk * 8) * 2;
    if constexpr (MAP) addr[p] = base[p] + from;
    else off[p] = (uint32_t)from;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + wave * PER * 1024;
  // by hand: the compiler would count these loads into what a wait for an LDS read waits for
  auto fetch = [&](int p, int slot, int advance) {
    if constexpr (MAP) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds0 + slot * SLOT + p * 1024), "v"(addr[p]) : "memory");
      addr[p] += advance;
    } else {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + slot * SLOT + p * 1024), "v"(off[p]), "s"(base[p]) : "memory");
      base[p] += advance;
    }
  };
  f32x4_t acc[NF][MF];
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int i = 0; i < MF; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // operand (row lane % 16, 16 bytes lane / 16 of a 32-element half): half 1 is half 0's address with bit 6 flipped
  const int f0 = (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) * 16), f1 = f0 ^ 64;
  const unsigned char* xb = lds + wm * MF * 2048;
  const unsigned char* wb = lds + (BM / 16 + wn * NF) * 2048;
#pragma unroll
  for (int p = 0; p < PER; ++p) fetch(p, 0, steps > 1 ? LT_BK * 2 : 0);
#pragma unroll
  for (int p = 0; p < PER; ++p) fetch(p, 1, steps > 2 ? LT_BK * 2 : 0);
  u32x4_t xf[MF], wa[NF], wd[NF];
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < NF; ++j) wa[j] = *reinterpret_cast<const u32x4_t*>(wb + f0 + j * 2048);
#pragma unroll
  for (int i = 0; i < MF; ++i) xf[i] = *reinterpret_cast<const u32x4_t*>(xb + f0 + i * 2048);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): scalar loads still in flight would make every wait for an LDS read this one
  for (int k = 0; k < steps; ++k) {
    const int here = (k & 1) * SLOT, next = SLOT - here;
#pragma unroll
    for (int j = 0; j < NF; ++j) wd[j] = *reinterpret_cast<const u32x4_t*>(wb + here + f1 + j * 2048);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MF; ++i) {
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[j][i] = mfma_bf16(wa[j], xf[i], acc[j][i]);
      xf[i] = *reinterpret_cast<const u32x4_t*>(xb + here + f1 + i * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next slot has landed (its loads are a step old) and this one has been read, here and after the barrier everywhere
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < NF; ++j) wa[j] = *reinterpret_cast<const u32x4_t*>(wb + next + f0 + j * 2048);
    __builtin_amdgcn_sched_barrier(0);
    const int advance = k + 3 < steps ? LT_BK * 2 : 0;
#pragma unroll
    for (int i = 0; i < MF; ++i) {
#pragma unroll
      for (int p = i * PER / MF; p < (i + 1) * PER / MF; ++p) fetch(p, k & 1, advance);
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[j][i] = mfma_bf16(wd[j], xf[i], acc[j][i]);
      xf[i] = *reinterpret_cast<const u32x4_t*>(xb + next + f0 + i * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // epilogue, EI row operands at a time: the wave's sums through LDS of its own, so that a lane then takes 4 neighbouring columns of a row and
  // 4 * NF lanes a whole run of them
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();                               // every wave has read its last operands, and no load is on its way into LDS
  constexpr int EI = MF / 2, LDT = 16 * NF + 4, LPR = 4 * NF / HALVES, RPP = 64 / LPR;   // (lanes per row, rows per pass)
  float* tile_lds = reinterpret_cast<float*>(lds) + wave * (EI * 16 * LDT);
#pragma unroll
  for (int i0 = 0; i0 < MF; i0 += EI) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < EI; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j)
        *reinterpret_cast<f32x4_t*>(tile_lds + (i * 16 + (lane & 15)) * LDT + j * 16 + (lane >> 4) * 4) = acc[j][i0 + i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int n = n0 + wn * WCOLS + (lane % LPR) * 4;
    f32x4_t b;
    if constexpr (!GATED) b = lin_bias4(a, g, n, vec4);
#pragma unroll 1
    for (int r0 = 0; r0 < EI * 16; r0 += RPP) {
      const int row = r0 + lane / LPR, t = m0 + (wm * MF + i0) * 16 + row;
      if (t >= t_hi || n >= a.N) continue;
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(tile_lds + row * LDT + (lane % LPR) * 4);
      // parts: [part][row][group][column], padded to whole 4 columns (GATED: the sums with w and w2 as two groups)
      const int n4 = (a.N + 3) & ~3;
      if constexpr (GATED) {
        const f32x4_t u = *reinterpret_cast<const f32x4_t*>(tile_lds + row * LDT + WCOLS + (lane % LPR) * 4);
        if (parts == 1) {
          lin_gated4(a, t, n, v, u, vec4);
        } else {
          float* to = slab + ((size_t)part * a.T + t) * 2 * n4 + n;
          *reinterpret_cast<f32x4_t*>(to) = v;
          *reinterpret_cast<f32x4_t*>(to + n4) = u;
        }
      } else if (parts == 1) {
        lin_epilogue4(a, g, t, n, v, b, vec4);
      } else {
        *reinterpret_cast<f32x4_t*>(slab + (((size_t)part * a.T + t) * gridDim.y + g) * n4 + n) = v;
      }
    }
  }
}

// the K parts of every element in order, then the epilogue: 4 columns per thread
__global__ __launch_bounds__(256) void linear_parts_kernel(LinArgs a, int groups, int parts, const float* slab, bool vec4) {
  const int n4 = (a.N + 3) & ~3, quads = n4 / 4;
  const size_t total = (size_t)a.T * groups * quads;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(slab + e * 4);
    for (int p = 1; p < parts; ++p) v += *reinterpret_cast<const f32x4_t*>(slab + ((size_t)p * total + e) * 4);
    const int n = (int)(e % quads) * 4;
    const size_t q = e / quads;
    const int g = (int)(q % groups), t = (int)(q / groups);
    lin_epilogue4(a, g, t, n, v, lin_bias4(a, g, n, vec4), vec4);
  }
}

// the same for the gated form
__global__ __launch_bounds__(256) void linear_gated_parts_kernel(LinArgs a, int parts, const float* slab, bool vec4) {
  const int n4 = (a.N + 3) & ~3, quads = n4 / 4;
  const size_t total = (size_t)a.T * quads, step = (size_t)a.T * 2 * n4;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const int n = (int)(e % quads) * 4, t = (int)(e / quads);
    const float* from = slab + (size_t)t * 2 * n4 + n;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(from), u = *reinterpret_cast<const f32x4_t*>(from + n4);
    for (int p = 1; p < parts; ++p) {
      v += *reinterpret_cast<const f32x4_t*>(from + p * step);
      u += *reinterpret_cast<const f32x4_t*>(from + p * step + n4);
    }
    lin_gated4(a, t, n, v, u, vec4);
  }
}

template <int MF, int NF, int WM, int WN, bool MAP, bool GATED = false>
int go(const LinArgs& a, const LinTilePlan& p, int Tg, int groups, float* slab, hipStream_t s) {
  constexpr int BM = 16 * MF * WM, BN = 16 * NF * WN, RING = LT_SLOTS * (BM + BN) * LT_BK * 2;
  constexpr int EPI = WM * WN * (MF / 2) * 16 * (16 * NF + 4) * 4, LDS = RING > EPI ? RING : EPI;
  auto kern = linear_pipe_kernel<MF, NF, WM, WN, MAP, GATED>;
  // the grant is per device: asked for at every launch (a lookup in the runtime)
  if (LDS > 64 * 1024)
    DIHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS), DIHIP_RUNTIME_ERROR);
  const int mt = (Tg + BM - 1) / BM, nt = GATED ? (a.N + BN / 2 - 1) / (BN / 2) : (a.N + BN - 1) / BN;
  const bool vec4 = lin_vec4(a);
  // (segments: as many row tiles as T rows in `groups` segments of at most Tg can need)
  const dim3 grid(a.seg ? (unsigned)nt * (unsigned)(mt * (long)groups < a.T / BM + groups ? mt * groups : a.T / BM + groups) : mt * nt, a.seg ? 1 : groups, p.parts);
  hipLaunchKernelGGL(kern, grid, dim3(64 * WM * WN), LDS, s, a, mt, nt, groups, vec4, p.parts, slab);
  if (p.parts > 1) {
    const size_t quads = (size_t)a.T * groups * ((a.N + 3) / 4);
    const dim3 pgrid((unsigned)((quads + 255) / 256 < 4096 ? (quads + 255) / 256 : 4096));
    if constexpr (GATED) hipLaunchKernelGGL(linear_gated_parts_kernel, pgrid, dim3(256), 0, s, a, p.parts, slab, vec4);
    else hipLaunchKernelGGL(linear_parts_kernel, pgrid, dim3(256), 0, s, a, groups, p.parts, slab, vec4);
  }
  return launch_status();
}

}  // namespace

// Which tile, and into how many parts K is split: the shortest of (rounds over the CUs) x (steps of a part) x (time of a step) + the slab's way
// through memory.  192 x 256 is there for row counts that the others cut badly: 513 rows 14336 -> 4096 take 100.7 us in 128 x 128, 102.7 in 256 x 256
// and 91.3 in 192 x 256; 300 rows 4096 -> 14336 82 / 85 / 74.5; 1500 rows 226 / 208 / 193.  (256 x 224 and 256 x 192, which fill the last round better at
// some widths, gave 2 % at 2048 rows: the clock falls as the chip fills.)  A launch with its prologue 5 us, the launch that adds parts 4 us and the slab's
// bytes, out and in, at 4.5 TB/s.  Over 65 .. 2048 rows and 512 .. 32000 columns (100 products) the choice is on average 0.5 % behind the best of the three tiles, at
// worst 13 %; unsplit, 513 rows 8192 -> 2048 take 107 us instead of 39.  The parts follow the row count, and with them the order of an element's f32 sums.
struct TileShape {
  int bm, bn;
  double step_us;   // of 64 of K, on every CU at once.  128 x 128: for one workgroup per CU (two at a time: TWO_SMALL_US)
};
constexpr TileShape SHAPES[] = {{256, 256, 1.70}, {192, 256, 1.47}, {128, 128, 0.9}};
constexpr int SMALL = 2;
constexpr double TWO_SMALL_US = 1.2;
LinTilePlan plan_linear_tile(int Tg, int N, int K, int groups, long ldx, bool split) {
  LinTilePlan best{};
  // (a tile's rows of w, and of x where no map names them, are addressed with 32-bit offsets)
  if (K % LT_BK || K <= 0 || (size_t)256 * (size_t)K * 2 >= (1ull << 31) || (size_t)256 * (size_t)ldx * 2 >= (1ull << 31)) return best;
  constexpr size_t MOST = (size_t)192 << 20;   // of slab
  constexpr int ncu = 256;
  const int all = K / LT_BK;
  double best_us = 0;
  for (int sh = 0; sh <= SMALL; ++sh) {
    const long tiles = (long)((Tg + SHAPES[sh].bm - 1) / SHAPES[sh].bm) * ((N + SHAPES[sh].bn - 1) / SHAPES[sh].bn) * groups;
    for (int p = 1; p <= (split ? 16 : 1); ++p) {
      if (p > 1 && (all / p < 4 || tiles * p > 2 * ncu)) break;
      const size_t slab = p > 1 ? (size_t)p * Tg * groups * ((N + 3) & ~3) * sizeof(float) : 0;
      if (slab > MOST) break;
      const long wgs = tiles * p;
      const double round_us = sh == SMALL && wgs > ncu ? TWO_SMALL_US * ((wgs + 2 * ncu - 1) / (2 * ncu)) : SHAPES[sh].step_us * ((wgs + ncu - 1) / ncu);
      const double us = round_us * ((all + p - 1) / p) + 5 + (p > 1 ? 4 + 2.0 * slab / 4.5e6 : 0);
      if (!best.ok || us < best_us) {
        best = LinTilePlan{true, sh, p, slab};
        best_us = us;
      }
    }
  }
  return best;
}

int launch_linear_tile(const LinArgs& a, const LinTilePlan& p, int Tg, int groups, float* slab, hipStream_t s) {
  DIHIP_REQUIRE(groups <= 65535, DIHIP_PARAM_ERROR, "linear: more than 65535 groups");
  if (a.w2) {
    switch (p.shape) {
      case 0: return go<8, 4, 2, 4, false, true>(a, p, Tg, 1, slab, s);
      case 1: return go<6, 4, 2, 4, false, true>(a, p, Tg, 1, slab, s);
      default: return go<4, 4, 2, 2, false, true>(a, p, Tg, 1, slab, s);
    }
  }
  if (a.row_map) {
    switch (p.shape) {
      case 0: return go<8, 4, 2, 4, true>(a, p, Tg, groups, slab, s);
      case 1: return go<6, 4, 2, 4, true>(a, p, Tg, groups, slab, s);
      default: return go<4, 4, 2, 2, true>(a, p, Tg, groups, slab, s);
    }
  }
  switch (p.shape) {
    case 0: return go<8, 4, 2, 4, false>(a, p, Tg, groups, slab, s);
    case 1: return go<6, 4, 2, 4, false>(a, p, Tg, groups, slab, s);
    default: return go<4, 4, 2, 2, false>(a, p, Tg, groups, slab, s);
  }
}

}  // namespace dihip
