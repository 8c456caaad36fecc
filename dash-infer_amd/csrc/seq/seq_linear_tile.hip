// seq_linear_tile.hip -- linear_pipe_kernel: products of many bf16 rows (prompts, portions) with bf16 weights, on the matrix cores.
//
// A workgroup of 8 waves owns a tile (256 x 256 down to 64 x 128) and walks K in steps of 64 through two rings of LDS slots, one for rows, one for weights:
//   * rows and weights go straight into LDS (global_load_lds, 16 bytes a lane): no registers and no instructions for staging.  A 1 KiB piece is 8
//     rows x 128 bytes in the order of the lanes (whole cache lines: with 64-byte pieces the L2s had twice the requests, 236 against
//     226 us), so the 16-byte chunks of a row change places on the memory side (chunk ^ row % 8) and the operand reads of 8
//     consecutive lanes touch every bank once;
//   * weights come from HBM, and one step (1 .. 1.5 us) is no longer than such a load takes: they are asked for three or four steps ahead, rows, which the L2s hold,
//     two to four.  The largest tile takes all of the 160 KB (2 slots of rows, 3 of weights).  With two slots of both, weights not in any cache: 2048 rows 4096 -> 14336 twice
//     436 -> 405 us, 14336 -> 4096 209 -> 194, 700 rows 4096 -> 14336 twice 197 -> 164, 513 rows 2048 -> 6208 35 -> 22;
//   * a step is two halves of 32.  While the first multiplies, the operands of the second are read; then one barrier tells that these slots have
//     been read and the next ones have landed; while the second half multiplies, the slots are
//     refilled and the next step's first operands are read.  The tail re-reads the last step instead of branching;
//   * the order of products, reads and loads is pinned (sched_barrier): left alone the compiler moves the reads behind the products;
//   * the loads are inline asm (they return nothing into registers): the compiler would count them into every wait for an LDS read.
// 2048 rows, 4096 -> 28672 run at 1 190 TFLOP/s; the matrix pipes' clock is 2.0 GHz there, and 3.5 rounds of tiles take the time of 4.
// One wave per SIMD with 128 x 128 each, which reads half as much LDS per product, was twice as slow (sums in both register files, copied to and fro).
//
// Narrow outputs and short prompts have too few tiles for 256 CUs: K is then split over workgroups that leave f32 tiles in a slab,
// and linear_parts_kernel adds them in order (plan_linear_tile).
#include "seq_linear.h"
#include <cmath>

namespace dihip {
namespace {

constexpr int LT_BK = 64;

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
// cost beside the products: f32 sums out and in again, and the last round of tiles twice (with two slots of LDS each: 2048 rows 4096 -> 14336 twice 491 -> 444 us, 1500
// rows 423 -> 334; 2048 -> 8192 twice, 513 rows 92.7 -> 58.2, 128 rows 44.8 -> 28.7).
// SX / SW: LDS slots (steps of 64) of the rows and of the weights
template <int MF, int NF, int WM, int WN, int SX, int SW, bool MAP, bool GATED>
__global__ __launch_bounds__(64 * WM * WN, (WM * WN) / 4) void linear_pipe_kernel(LinArgs a, int mtiles, int ntiles, int groups, bool vec4, int parts, float* slab) {
  constexpr int WAVES = WM * WN, BM = 16 * MF * WM, BN = 16 * NF * WN;
  constexpr int PX = (BM / 8 + WAVES - 1) / WAVES, PW = BN / 8 / WAVES, PER = PX + PW;   // 1 KiB pieces (8 rows x 128 bytes) of a K step, per wave
  static_assert(BN / 8 % WAVES == 0 && (SW == SX || SW == SX + 1), "whole pieces of weights per wave; what the waits count on");
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
  const char* wfrom = GATED && wave * PW * 8 % (2 * WCOLS) >= WCOLS ? w2base : wbase;
  uint32_t xoffs[PX], woffs[PW];   // (the host checks that 256 rows lie within 2 GB)
  const char* xaddr[PX];           // (MAP, instead of xoffs)
  int xpiece[PX];
#pragma unroll
  for (int p = 0; p < PX; ++p) {
    xpiece[p] = BM / 8 % WAVES ? min(wave * PX + p, BM / 8 - 1) : wave * PX + p;   // (the last may come twice)
    const int r = min(m0 + xpiece[p] * 8 + prow, t_hi - 1);
    const size_t from = ((MAP ? (size_t)a.row_map[r] : (size_t)(r - m0)) * (size_t)a.ldx + pchunk * 8) * 2;
    if constexpr (MAP) xaddr[p] = xbase + from;
    else xoffs[p] = (uint32_t)from;
  }
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    int wrow = (wave * PW + p) * 8;
    if constexpr (GATED) wrow = wrow / (2 * WCOLS) * WCOLS + wrow % WCOLS;
    woffs[p] = (uint32_t)(((size_t)min(wrow + prow, a.N - 1 - n0) * a.K + pchunk * 8) * 2);
  }
  constexpr int XSLOT = BM * 128, WSLOT = BN * 128, WRING = SX * XSLOT;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  // by hand: the compiler would count these loads into what a wait for an LDS read waits for
  auto fetch_x = [&](int p, int slot, int advance) {
    const uint32_t to = lds0 + slot * XSLOT + xpiece[p] * 1024;
    if constexpr (MAP) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(xaddr[p]) : "memory");
      xaddr[p] += advance;
    } else {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(xoffs[p]), "s"(xbase) : "memory");
      if (p == PX - 1) xbase += advance;
    }
  };
  auto fetch_w = [&](int p, int slot, int advance) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + WRING + slot * WSLOT + (wave * PW + p) * 1024), "v"(woffs[p]), "s"(wfrom) : "memory");
    if (p == PW - 1) wfrom += advance;
  };
  auto fetch = [&](int p, int xslot, int xadvance, int wslot, int wadvance) {
    if (p < PX) fetch_x(p, xslot, xadvance);
    else fetch_w(p - PX, wslot, wadvance);
  };
  f32x4_t acc[NF][MF];
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int i = 0; i < MF; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // operand (row lane % 16, 16 bytes lane / 16 of a 32-element half): half 1 is half 0's address with bit 6 flipped
  const int f0 = (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) * 16), f1 = f0 ^ 64;
  const unsigned char* xb = lds + wm * MF * 2048;
  const unsigned char* wb = lds + WRING + wn * NF * 2048;
  // in the order of the steps: rows, then weights, which are SW - SX steps ahead of them
  if constexpr (SW > SX)
#pragma unroll
    for (int p = 0; p < PW; ++p) fetch_w(p, 0, steps > 1 ? LT_BK * 2 : 0);
#pragma unroll
  for (int q = 0; q < SX; ++q)
#pragma unroll
    for (int p = 0; p < PER; ++p) fetch(p, q, q + 1 < steps ? LT_BK * 2 : 0, q + SW - SX, q + 1 + SW - SX < steps ? LT_BK * 2 : 0);
  constexpr int AHEAD = SW > SX ? PW : 0;   // of the loads behind those of a step's rows: weights of a later step
  u32x4_t xf[MF], wa[NF], wd[NF];
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD + (SX - 1) * PER) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < NF; ++j) wa[j] = *reinterpret_cast<const u32x4_t*>(wb + f0 + j * 2048);
#pragma unroll
  for (int i = 0; i < MF; ++i) xf[i] = *reinterpret_cast<const u32x4_t*>(xb + f0 + i * 2048);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): scalar loads still in flight would make every wait for an LDS read this one
  int xs = 0, ws = 0;   // the slots of step k
  for (int k = 0; k < steps; ++k) {
    const int xs1 = xs + 1 == SX ? 0 : xs + 1, ws1 = ws + 1 == SW ? 0 : ws + 1;
#pragma unroll
    for (int j = 0; j < NF; ++j) wd[j] = *reinterpret_cast<const u32x4_t*>(wb + ws * WSLOT + f1 + j * 2048);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MF; ++i) {
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[j][i] = mfma_bf16(wa[j], xf[i], acc[j][i]);
      xf[i] = *reinterpret_cast<const u32x4_t*>(xb + xs * XSLOT + f1 + i * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next slot has landed (its loads are a step old) and this one has been read, here and after the barrier everywhere
    asm volatile("" ::: "memory");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(AHEAD + (SX - 2) * PER) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < NF; ++j) wa[j] = *reinterpret_cast<const u32x4_t*>(wb + ws1 * WSLOT + f0 + j * 2048);
    __builtin_amdgcn_sched_barrier(0);
    const int xadvance = k + 1 + SX < steps ? LT_BK * 2 : 0, wadvance = k + 1 + SW < steps ? LT_BK * 2 : 0;
#pragma unroll
    for (int i = 0; i < MF; ++i) {
#pragma unroll
      for (int p = i * PER / MF; p < (i + 1) * PER / MF; ++p) fetch(p, xs, xadvance, ws, wadvance);
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[j][i] = mfma_bf16(wd[j], xf[i], acc[j][i]);
      xf[i] = *reinterpret_cast<const u32x4_t*>(xb + xs1 * XSLOT + f0 + i * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
    xs = xs1;
    ws = ws1;
  }
  // epilogue, EI row operands at a time: the wave's sums through LDS of its own, so that a lane then takes 4 neighbouring columns of a row and
  // 4 * NF lanes a whole run of them
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();                               // every wave has read its last operands, and no load is on its way into LDS
  constexpr int EI = (MF + 1) / 2, LDT = 16 * NF + 4, LPR = 4 * NF / HALVES, RPP = 64 / LPR;   // (lanes per row, rows per pass)
  float* tile_lds = reinterpret_cast<float*>(lds) + wave * (EI * 16 * LDT);
#pragma unroll
  for (int i0 = 0; i0 < MF; i0 += EI) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < EI; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j)
        if (i0 + i < MF) *reinterpret_cast<f32x4_t*>(tile_lds + (i * 16 + (lane & 15)) * LDT + j * 16 + (lane >> 4) * 4) = acc[j][i0 + i < MF ? i0 + i : 0];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int n = n0 + wn * WCOLS + (lane % LPR) * 4;
    f32x4_t b;
    if constexpr (!GATED) b = lin_bias4(a, g, n, vec4);
#pragma unroll 1
    for (int r0 = 0; r0 < EI * 16; r0 += RPP) {
      const int row = r0 + lane / LPR, t = m0 + (wm * MF + i0) * 16 + row;
      if (t >= t_hi || n >= a.N || (MF % 2 && i0 * 16 + row >= MF * 16)) continue;
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
        lin_epilogue4<!MAP>(a, g, t, n, v, b, vec4);
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

template <int MF, int NF, int WM, int WN, int SX, int SW, bool MAP, bool GATED>
int go(const LinArgs& a, const LinTilePlan& p, int Tg, int groups, float* slab, hipStream_t s) {
  constexpr int BM = 16 * MF * WM, BN = 16 * NF * WN, RING = (SX * BM + SW * BN) * LT_BK * 2;
  constexpr int EPI = WM * WN * ((MF + 1) / 2) * 16 * (16 * NF + 4) * 4, LDS = RING > EPI ? RING : EPI;
  auto kern = linear_pipe_kernel<MF, NF, WM, WN, SX, SW, MAP, GATED>;
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

// Which tile, and into how many parts K is split: the shortest of (rounds over the CUs) x (steps of a part x time of a step + a tile's prologue and way out), bounded by
// the weights' way from HBM, + the slab's way through memory.  The constants are a fit to 143 products (65 .. 2048 rows, 512 .. 14336 -> 512 .. 28672 columns) with
// every tile in 1 .. 8 parts, weights not in any cache; over those the choice is on average 1.8 % behind the best of them, at worst 20 % (12 us of a launch), and 0.86 of
// the time of three tiles (256 x 256, 192 x 256, 128 x 128) with two slots each.  The many heights are for row counts that others cut badly: 513 rows 4096 -> 28672 145 us in 160 x 256
// (164 in 192 x 256), 300 rows 2048 -> 16384 32.3 in 160 x 128 (43.8), 513 rows 2048 -> 6208 22.6 in 128 x 128 (34.7), 2048 rows 4096 -> 4096 62 in 256 x 128 (78), 200 rows
// 2048 -> 2048 12.5 in 64 x 128 (18.7).  The parts follow the row count, and with them the order of an element's f32 sums.
struct TileShape {
  int bm, bn;
  double step_us;   // of 64 of K, on every CU at once
};
constexpr TileShape SHAPES[] = {{256, 256, 1.33}, {224, 256, 1.23}, {192, 256, 1.09}, {160, 256, .95}, {128, 256, .82}, {256, 128, .78},
                                {192, 128, .62}, {160, 128, .57}, {128, 128, .485}, {96, 128, .413}, {64, 128, .331}};
LinTilePlan plan_linear_tile(int Tg, int N, int K, int groups, long ldx, bool split, bool gated) {
  LinTilePlan best{};
  const int cols = gated ? 2 * N : N;
  const size_t slab_part = lin_slab_part_bytes(Tg, N, gated ? 2 : groups);
  // (a tile's rows of w, and of x where no map names them, are addressed with 32-bit offsets)
  if (K % LT_BK || K <= 0 || (size_t)256 * (size_t)K * 2 >= (1ull << 31) || (size_t)256 * (size_t)ldx * 2 >= (1ull << 31)) return best;
  constexpr size_t MOST = (size_t)192 << 20;   // of slab
  constexpr double LAUNCH_US = 2.5, TILE_US = 3.9, PARTS_US = 4.0, PART_US = 0.6, SLAB_BYTES_PER_US = 5.5e6, HBM_BYTES_PER_US = 4.6e6;
  constexpr int ncu = 256;
  const int all = K / LT_BK;
  const double hbm_us = 2.0 * K * (double)cols * groups / HBM_BYTES_PER_US, hbm4 = hbm_us * hbm_us * hbm_us * hbm_us;
  double best_us = 0;
  for (int sh = 0; sh < (int)(sizeof(SHAPES) / sizeof(SHAPES[0])); ++sh) {
    const long tiles = (long)((Tg + SHAPES[sh].bm - 1) / SHAPES[sh].bm) * ((cols + SHAPES[sh].bn - 1) / SHAPES[sh].bn) * groups;
    for (int p = 1; p <= (split ? 16 : 1); ++p) {
      if (p > 1 && (all / p < 4 || tiles * p > 2 * ncu)) break;
      const size_t slab = p > 1 ? p * slab_part : 0;
      if (slab > MOST) break;
      const double body = (SHAPES[sh].step_us * ((all + p - 1) / p) + TILE_US) * ((tiles * p + ncu - 1) / ncu);
      const double us = LAUNCH_US + std::sqrt(std::sqrt(body * body * body * body + hbm4)) + (p > 1 ? PARTS_US + PART_US * p + 2.0 * slab / SLAB_BYTES_PER_US : 0);
      if (!best.ok || us < best_us) {
        best = LinTilePlan{true, sh, p, slab};
        best_us = us;
      }
    }
  }
  return best;
}

namespace {
template <bool MAP, bool GATED>
int go_shape(const LinArgs& a, const LinTilePlan& p, int Tg, int groups, float* slab, hipStream_t s) {
  switch (p.shape) {   // (as SHAPES)
    case 0: return go<8, 4, 2, 4, 2, 3, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 1: return go<7, 4, 2, 4, 2, 3, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 2: return go<6, 4, 2, 4, 2, 3, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 3: return go<5, 4, 2, 4, 3, 3, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 4: return go<4, 4, 2, 4, 3, 3, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 5: return go<8, 2, 2, 4, 3, 3, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 6: return go<6, 2, 2, 4, 3, 4, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 7: return go<5, 2, 2, 4, 3, 4, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 8: return go<4, 2, 2, 4, 4, 4, MAP, GATED>(a, p, Tg, groups, slab, s);
    case 9: return go<3, 2, 2, 4, 4, 4, MAP, GATED>(a, p, Tg, groups, slab, s);
    default: return go<2, 2, 2, 4, 4, 4, MAP, GATED>(a, p, Tg, groups, slab, s);
  }
}
}  // namespace

int launch_linear_tile(const LinArgs& a, const LinTilePlan& p, int Tg, int groups, float* slab, hipStream_t s) {
  DIHIP_REQUIRE(groups <= 65535, DIHIP_PARAM_ERROR, "linear: more than 65535 groups");
  if (a.w2) return go_shape<false, true>(a, p, Tg, 1, slab, s);
  return a.row_map ? go_shape<true, false>(a, p, Tg, groups, slab, s) : go_shape<false, false>(a, p, Tg, groups, slab, s);
}

}  // namespace dihip
