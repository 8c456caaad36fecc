// gemm_prefill_kernel.hpp -- weight-only (A16W8 / A16W4) GEMM for the CONTEXT phase (M >= 64 rows) on gfx950.
//
// The general kernel (gemm_lowp_kernel.hpp) keeps at most 32 activation rows per workgroup: a 2048-token prompt walks every
// weight matrix 64 times and the context phase of Qwen2-7B ran at 9 % of the dense bf16 MFMA peak (profiles/r03f_bench_prefill_2048.json:
// 119 ms, of which the attention is 1.5).  This kernel is the large-M member of the family -- replaces, for prefill shapes,
// the reference's dequantise + cuBLAS fall-back and its 16816 tensor-core kernels (gemm_a16w8_kernel.h:239-331,
// hgemm_a16w4_subc_32x256x32, gemm_a16w4_subc_kernel.cu:466-815):
//
//   * workgroup tile 128 rows (or 112, 96, 80: TR) x 256 columns (8 waves side by side in N, each 128 x 32 = 8 row tiles x 2 column tiles of
//     v_mfma_f32_16x16x32: 16 accumulators), K walked in packed k-tiles (W4: 128 k, W8: 64 k, two of them where no group
//     ends in between);
//   * A (activations, FT row-major) goes straight from memory into LDS (global_load_lds: no registers, no instructions for staging),
//     double-buffered: the loads of k-tile t + 1 are in flight while t is multiplied, ONE barrier per k-tile; every wave reads all
//     row tiles;
//   * B (weights) never touches LDS: "dihip tile-major" packing makes a lane's 16-byte load the B fragment of its own column
//     tile (x KSTEPS), and no two waves share a column tile;
//   * the same exact-integer arithmetic as the decode kernels: q expands to 128 + q in FT with the magic-number trick, the MFMA
//     sums exact products, and per quantisation group  y += s * (acc - (z + 128) * sum_k x)  on the f32 accumulator, with
//     sum_k x per (row, k-tile) taken under the multiply -- an MFMA against a fragment of ones per wave and k-step;
//   * the fix-up of a closed group runs under the first products of the next one, row tile by row tile (vector instructions
//     while the matrix unit works), and so do the expansions of the next k-step's weights;
//   * epilogues as everywhere: STD (alpha, bias, UnaryType activation, FT residual), SwiGLU over a gate / up pair (a wave's two
//     column tiles are then the SAME 16 columns of the two matrices: 128 output columns per workgroup), f32 hidden-stream update.
//
// Host contract (gemm_lowp.hip: run_gemm): bf16 / f16 activations row-major with ldx % 8 == 0, 16-byte aligned; K a multiple of
// the k-tile; group_size a multiple of the k-tile or per-channel.  Rows >= M are clamped on load and masked on store.
//
// What bounds it (gate / up pair of 2048 rows, K = 3584, 2 x 18944 columns, W4 in groups of 128; counters): 240 registers mean one
// workgroup = two waves per SIMD.  Per wave and k-tile 68 MFMAs of 16 cycles, about 190 other vector and 45 LDS instructions; the LDS
// reads (256 KiB per k-tile) alone take the products' time once.  The matrix units are busy 44 % of the time at 2.05 GHz; timing copies
// of the kernel with one part left out: - 16 % without the fix-up, - 13 % without the row sums, - 14 % without the loads, - 5 % without the
// expansions, - 10 % without the LDS reads of all but the first k-step, - 44 % without all of them (1 600 TFLOP/s).  The parts add up:
// what is left is instruction issue and power, not one wait.
// Measured: 2048 rows of four W4 layers 5.29 ms with A through registers and the fix-up between the tiles, 5.05 as above, 4.86 with four
// neighbouring columns per lane and an epilogue without branches; 326 rows of four W8 layers 1.76 -> 1.63 ms, 1.33 on tiles of
// 112 rows with two k-tiles between two barriers.
// A 2 x 4 grid of waves with 64 x 64 tiles (half the LDS reads, twice the expansions and twice the weight loads) made those four layers 6 % slower.
#pragma once
#include <atomic>
#include <type_traits>
#include "gemm_lowp_kernel.hpp"
#include "gemv_stream_kernel.hpp"  // ExpandV: the 128 + q expansion of the decode kernels

namespace dihip {

constexpr int PF_WAVES = 8;
constexpr int PF_THREADS = PF_WAVES * 64;
constexpr int PF_BM = 128;           // rows per workgroup at most (8 row tiles; PrefillArgs::bm, the kernel's TR: how many it takes)
constexpr int PF_WM = 1;             // waves along M
constexpr int PF_WN = PF_WAVES / PF_WM;
constexpr int PF_TR = PF_BM / 16;    // row tiles of the workgroup at most (= waves: wave w stages row tile w)
constexpr int PF_TR_LEAST = 5;       // ... and at least
constexpr int PF_CW = 2 * PF_WM;     // column tiles per wave (the workgroup covers 256 columns either way)
static_assert(PF_TR == PF_WAVES && PF_WM == 1, "one staged row tile per wave, every wave all of them");
static_assert(PF_CW == 2, "the two column tiles of a wave are named one by one where the sums change hands");

struct PrefillArgs {
  const u32x4_t* w0;
  const u32x4_t* w1;    // EPI_SWIGLU: "up" weight
  const uint32_t* sz0;  // [NTILES][Gp][16] (scale | zero << 16)
  const uint32_t* sz1;
  const void* x;        // FT [M, ldx]
  int ldx;
  const void* bias;
  const void* residual;  // FT [M, ldy]
  void* y;               // FT [M, ldy]
  int ldy;
  const float* h_res;  // EPI_ADDTO
  float* h_out;
  float alpha;
  int act;
  int M, N;
  int KT;      // k-tiles
  int NTILES;  // 16-column tiles
  int Gp;      // (scale, zero) groups stored per tile
  int ktpg;    // k-tiles per quantisation group (per-channel: >= KT)
  int col_blocks;
  int bm;      // rows per workgroup: 16 * TR of the kernel
  // Split in K: column blocks [tail_cb, col_blocks) -- the workgroups that would otherwise run as a last, mostly empty
  // round on the chip (qkv of Qwen2-7B at 2048 rows: 288 tiles on 256 CUs), or all of them where the whole grid fills at most half
  // of it (short prompts) -- are walked by `ksplit` workgroups each, one K range apiece (whole quantisation groups; the ranges
  // differ by at most one), which leave their f32 tile in `slab`; gemm_prefill_tail_reduce_kernel adds the parts in order and
  // applies the epilogue.  tail_cb == col_blocks: no split.
  int tail_cb;
  int ksplit;
  int kunit;    // k-tiles that a K range must not cut (grouped weights: a group; per-channel: 1, 8 bits where every tile is split: 2)
  int wide_out; // four neighbouring columns of an output (and residual) row make one aligned access
  float* slab;  // [tail tile][ksplit][bm][256] f32
};

template <int WBITS, int TR, int UK>
constexpr size_t prefill_lds_bytes() {
  // 2 x A tile (16 TR rows x UK KSTEPS x 64 bytes) + 2 x 128 row sums
  return (size_t)2 * TR * UK * WTraits<WBITS>::KSTEPS * 1024 + 2 * PF_BM * sizeof(float);
}

// (GPT -- one k-tile per quantisation group -- is a compile-time copy of the same code: the group test folds away)
// TR: row tiles of a workgroup, 5 .. 8 (gemm_lowp.hip: prefill_tail_plan).  Rows past M cost what the others do: 326 rows are three tiles of 112 as well as three of 128
// UK: k-tiles between two barriers.  8 bits: two where no group ends between them; of one with its two k-steps the wait, the first operand reads and the expansions before the first
// product were more than half of the time.  int8 per channel, 326 rows 3584 -> 18944 twice 131.7 -> 121.2 us, 18944 -> 3584 74.3 -> 66.7, 64 rows 59.4 -> 51.0 and 37.5 -> 35.1
template <int WBITS, int FT, int EPI, int GPT, int TR, int UK>
__global__ __launch_bounds__(PF_THREADS, 2) void gemm_prefill_kernel(const PrefillArgs a) {
  using WT = WTraits<WBITS>;
  using EX = ExpandV<WBITS, FT>;
  constexpr int KSTEPS = WT::KSTEPS;
  constexpr int KTILE = WT::KTILE, NKS = UK * KSTEPS;   // (NKS: k-steps of an iteration)
  static_assert(UK == 1 || !GPT, "a group of one k-tile ends in every one");
  constexpr bool DUAL = EPI == EPI_SWIGLU;
  constexpr bool LACE = GPT && WBITS == 4;  // fix-up under the first k-step's products (8 bits: two k-steps, no registers left for it)
  constexpr int PF_RT = TR, BM = 16 * TR;
  constexpr size_t ABYTES = (size_t)TR * NKS * 1024;  // one A tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* xsum = reinterpret_cast<float*>(smem + 2 * ABYTES);  // [2][PF_BM]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ni = lane & 15, kb = lane >> 4;
  const int wm = wave / PF_WN, wn = wave - wm * PF_WN;  // this wave's place in the PF_WM x PF_WN grid
  // consecutive workgroups share a column block (its weights stay hot in the L2s) and walk the rows
  const int mblocks = (a.M + BM - 1) / BM;
  int cb = blockIdx.x / mblocks, mb = blockIdx.x - cb * mblocks;
  int kt0 = 0, kt1 = a.KT, split_part = -1, split_tile = 0;  // this workgroup's k-tiles; tail split: its part and tile
  if (cb >= a.tail_cb) {  // (uniform) mb fastest, then the K part, then the column block: the 16 row blocks of a part share its weights
    const int idx = (int)blockIdx.x - a.tail_cb * mblocks;
    mb = idx % mblocks;
    const int t = idx / mblocks;
    split_part = t % a.ksplit;
    const int cbt = t / a.ksplit;
    cb = a.tail_cb + cbt;
    const int ku = GPT ? 1 : a.kunit, units = a.KT / ku;
    kt0 = split_part * units / a.ksplit * ku;
    kt1 = split_part + 1 == a.ksplit ? a.KT : (split_part + 1) * units / a.ksplit * ku;
    split_tile = cbt * mblocks + mb;
  }
  const int m0 = mb * BM;

  // ---- this wave's column tiles -------------------------------------------------------------------
  // STD / ADDTO: PF_CW consecutive tiles of the one matrix;  SwiGLU: PF_CW / 2 tiles of gate (c < PF_CW / 2) and the same of up
  constexpr int HCW = PF_CW / 2;
  int tile[PF_CW];
  bool tile_ok[PF_CW];
  // (buffer loads: bases in scalar registers, one lane offset for all)
  __amdgpu_buffer_rsrc_t wp[PF_CW], szp[PF_CW];
#pragma unroll
  for (int c = 0; c < PF_CW; ++c) {
    const int t = DUAL ? (cb * PF_WN + wn) * HCW + (c % HCW) : (cb * PF_WN + wn) * PF_CW + c;
    tile_ok[c] = t < a.NTILES;
    tile[c] = min(t, a.NTILES - 1);
    const bool second = DUAL && c >= HCW;
    wp[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4_t*>((second ? a.w1 : a.w0) + (size_t)tile[c] * a.KT * 64), 0, a.KT * 1024, 0x00020000);
    szp[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>((second ? a.sz1 : a.sz0) + (size_t)tile[c] * a.Gp * 16), 0, a.Gp * 64, 0x00020000);
  }

  // ---- A: wave w brings row tile w straight into LDS (global_load_lds: no registers, no instructions for staging), pieces of 8 rows x 128
  // bytes; the 16-byte chunks of a row change places on the memory side (chunk ^ row % 8): 8 consecutive lanes of an operand read then
  // touch every bank once.  Rows past M re-read the last row (masked on store)
  constexpr int HALVES = UK * KTILE / 64;                       // 64 k of all rows: TR * 2 KiB
  const int prow = lane >> 3, pchunk = (lane & 7) ^ prow;
  const char* abase = reinterpret_cast<const char*>(a.x) + (size_t)m0 * a.ldx * 2;
  uint32_t aoff[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) aoff[p] = (uint32_t)((size_t)min(wave * 16 + p * 8 + prow, a.M - 1 - m0) * a.ldx * 2 + pchunk * 16);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * 2048;
  auto load_a = [&](int kt, int buf) {
    if (TR < PF_TR && wave >= TR) return;   // (uniform)
#pragma unroll
    for (int hh = 0; hh < HALVES; ++hh) {
      const char* src = abase + (UK > 1 ? (size_t)min(kt + hh, a.KT - 1) * KTILE * 2 : (size_t)kt * KTILE * 2 + hh * 128);   // (past K: the last once more, times nothing)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + (uint32_t)(buf * ABYTES) + hh * (TR * 2048) + p * 1024),
                     "v"(aoff[p]), "s"(src) : "memory");
    }
  };
  static_assert(UK == 1 || KTILE == 64, "a half per k-tile");
  u32x4_t wreg[UK][PF_CW];
  u32x4_t szreg[PF_CW] = {};   // the running group's, of this lane's four columns of each tile
  auto load_b = [&](int kt) {
#pragma unroll
    for (int u = 0; u < UK; ++u)
#pragma unroll
      for (int c = 0; c < PF_CW; ++c)
        wreg[u][c] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wp[c], lane * 16, (UK > 1 ? min(kt + u, a.KT - 1) : kt) * 1024, 2));   // (2: nontemporal)
  };
  // operand (row ni of a row tile, 16 bytes kb of k-step ks)
  const int mine = TR < PF_TR ? min(wave, TR - 1) : wave;   // the row tile whose sums this wave takes (the last one's more than once)
  const int f0 = ni * 128 + ((kb ^ (ni & 7)) * 16), f1 = f0 ^ 64;
  auto aread = [&](const unsigned char* tile, int rt, int ks) {
    return *reinterpret_cast<const u32x4_t*>(tile + (ks >> 1) * (TR * 2048) + rt * 2048 + ((ks & 1) ? f1 : f0));
  };

  // acc: exact integer products of the running quantisation group (MFMA); tot: the scaled result.  The weights are the first operand: lane
  // (kb, ni) holds columns kb * 4 .. + 3 of a column tile, row ni of a row tile -- four neighbours of one row, stored together
  f32x4_t acc[PF_RT][PF_CW], tot[PF_RT][PF_CW];
  const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int rt = 0; rt < PF_RT; ++rt)
#pragma unroll
    for (int c = 0; c < PF_CW; ++c) acc[rt][c] = tot[rt][c] = zero4;
  uint32_t ex_mask = 0x000F000Fu, ex_magic = FT == DIHIP_BF16 ? 0x43004300u : 0x64006400u;
  asm volatile("" : "+v"(ex_mask), "+v"(ex_magic));
  // scale / zero-point of a closed group on the accumulators of one row tile, with the group's row sums
  f32x4_t s_[PF_CW], nz_[PF_CW];
  const float* xs = nullptr;
  auto open_fix = [&](int group) {
    xs = xsum + (group & 1) * PF_BM + wm * PF_RT * 16 + ni;
#pragma unroll
    for (int c = 0; c < PF_CW; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s_[c][r] = ft_bits_to_f32<FT>(szreg[c][r] & 0xFFFFu);
        nz_[c][r] = -(ft_bits_to_f32<FT>(szreg[c][r] >> 16) + EX::OFFSET);
      }
  };
  auto fix = [&](int rt, int c, float xv) {
#pragma unroll
    for (int r = 0; r < 4; ++r) tot[rt][c][r] = fmaf(s_[c][r], fmaf(nz_[c][r], xv, acc[rt][c][r]), tot[rt][c][r]);
  };
  auto load_sz = [&](int group) {
#pragma unroll
    for (int c = 0; c < PF_CW; ++c) szreg[c] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(szp[c], kb * 16, min(group, a.Gp - 1) * 64, 0));
  };

  // One barrier per k-tile.  Behind it: this tile (its loads are a k-tile old) is in LDS, the other buffer has been read, the row sums of the tile
  // before are there.  The next tile's loads go out, then the products: the first k-step's carry the fix-up of the group that the tile before
  // closed (one k-tile per group; longer groups are fixed up in one go, once per group), every row operand is re-read for the next k-step
  // right behind its last product, and the row sums of this tile (sum_k x: the staged row tile times a fragment of ones) are taken on the way.
  int gl = 0;                                                   // k-tiles of the running group done
  int grp = GPT ? kt0 : (a.ktpg < a.KT ? kt0 / a.ktpg : 0);     // running group (a K part starts on a group boundary)
  load_a(kt0, 0);
  load_b(kt0);
  const u32x4_t ones = FT == DIHIP_BF16 ? u32x4_t{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u}
                                  : u32x4_t{0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
  if constexpr (LACE) {   // the first tile closes a group of nothing: sums, scales and products 0
    if (tid < 2 * PF_BM) xsum[tid] = 0.f;
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): scalar loads still in flight would make every wait for an LDS read this one
  for (int kt = kt0, it = 0; kt < kt1; kt += UK, ++it) {
    const int buf = it & 1;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    u32x4_t wcur[UK][PF_CW];
#pragma unroll
    for (int c = 0; c < PF_CW; ++c) {
      asm volatile("" : "+v"(szreg[c]));   // here they are: nothing further down waits for loads again
#pragma unroll
      for (int u = 0; u < UK; ++u) {
        asm volatile("" : "+v"(wreg[u][c]));
        wcur[u][c] = wreg[u][c];
      }
    }
    const uint32_t second = UK == 1 || kt + 1 < kt1 ? ~0u : 0u;   // (uniform) an odd range's last k-tile has no neighbour
    const auto frag = [&](int c, int ks) {
      u32x4_t f = EX::frag(wcur[ks / KSTEPS][c], ks % KSTEPS, ex_mask, ex_magic);
      if (UK > 1 && ks >= KSTEPS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) f[r] &= second;
      }
      return f;
    };
    if constexpr (LACE) {
      open_fix(grp - 1);
    } else if (kt > kt0 && (GPT || gl == 0)) {                         // (uniform) the tile before closed its group
      open_fix(grp - 1);
#pragma unroll
      for (int rt = 0; rt < PF_RT; ++rt) {
        const float xv = xs[rt * 16];
#pragma unroll
        for (int c = 0; c < PF_CW; ++c) {
          fix(rt, c, xv);
          acc[rt][c] = zero4;
        }
      }
    }
    const int nkt = min(kt + UK, kt1 - 1);                      // past the end: once more the last, read by nobody
    load_a(nkt, buf ^ 1);
    load_b(nkt);
    load_sz(grp);
    const unsigned char* tile = smem + buf * ABYTES;
    u32x4_t af[PF_RT], bf[PF_CW], own;
    float xv = 0.f;
    if constexpr (LACE) xv = xs[0];
#pragma unroll
    for (int rt = 0; rt < PF_RT; ++rt) af[rt] = aread(tile, wm * PF_RT + rt, 0);
    own = aread(tile, mine, 0);
#pragma unroll
    for (int c = 0; c < PF_CW; ++c) bf[c] = frag(c, 0);
    f32x4_t sx = zero4;
    __builtin_amdgcn_sched_barrier(0);
    auto kstep = [&](int ks, auto first) {
      constexpr bool FIRST = decltype(first)::value;            // closes the group before
      u32x4_t bn[PF_CW];
#pragma unroll
      for (int rt = 0; rt < PF_RT; ++rt) {
        if constexpr (FIRST) {
          fix(rt, 0, xv);
          fix(rt, 1, xv);
          if (rt + 1 < PF_RT) xv = xs[(rt + 1) * 16];
          // (the products that start the next sums wait for the old sums to be used: one set of registers)
          asm volatile("" : "+v"(tot[rt][0]), "+v"(tot[rt][1]), "+v"(af[rt]));
        }
#pragma unroll
        for (int c = 0; c < PF_CW; ++c) acc[rt][c] = mfma16<FT>(bf[c], af[rt], FIRST ? zero4 : acc[rt][c]);
        if (ks + 1 < NKS) af[rt] = aread(tile, wm * PF_RT + rt, ks + 1);
        if (rt == 2) {
          u32x4_t one = ones;
          if (UK > 1 && ks >= KSTEPS) {
#pragma unroll
            for (int r = 0; r < 4; ++r) one[r] &= second;
          }
          sx = mfma16<FT>(one, own, sx);
          if (ks + 1 < NKS) own = aread(tile, mine, ks + 1);
        }
        if (ks + 1 < NKS && rt >= PF_RT - 1 - PF_CW && rt < PF_RT - 1) bn[rt - (PF_RT - 1 - PF_CW)] = frag(rt - (PF_RT - 1 - PF_CW), ks + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (ks + 1 < NKS) {
#pragma unroll
        for (int c = 0; c < PF_CW; ++c) bf[c] = bn[c];
      }
    };
    kstep(0, std::integral_constant<bool, LACE>{});
#pragma unroll
    for (int ks = 1; ks < NKS; ++ks) kstep(ks, std::false_type{});
    if (kb == 0 && (TR == PF_TR || wave < TR)) {   // the lane with kb == 0 of a row's lanes owns its entry: no race
      float* p = xsum + (grp & 1) * PF_BM + wave * 16 + ni;
      *p = GPT || gl == 0 ? sx[0] : *p + sx[0];
    }
    gl += UK;
    if (GPT || gl == a.ktpg || kt + UK >= kt1) {
      gl = 0;
      ++grp;
    }
  }
  // the last group; and nothing may be on its way into LDS when the workgroup leaves
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  open_fix(grp - 1);
#pragma unroll
  for (int rt = 0; rt < PF_RT; ++rt) {
    const float xv = xs[rt * 16];
#pragma unroll
    for (int c = 0; c < PF_CW; ++c) fix(rt, c, xv);
  }

  // ---- split in K: this part's f32 tile to the slab (rows / columns of the workgroup tile; SwiGLU: gate columns, then up) ----
  if (split_part >= 0) {  // (uniform)
    float* st = a.slab + ((size_t)split_tile * a.ksplit + split_part) * (BM * 256) + (size_t)(wm * PF_RT * 16 + ni) * 256;
#pragma unroll
    for (int rt = 0; rt < PF_RT; ++rt) {
      if (m0 + (wm * PF_RT + rt) * 16 >= a.M) break;  // (uniform) rows past M are never read
#pragma unroll
      for (int c = 0; c < PF_CW; ++c) {
        const int col = DUAL ? (c < HCW ? 0 : 128) + (wn * HCW + (c % HCW)) * 16 : (wn * PF_CW + c) * 16;
        *reinterpret_cast<f32x4_t*>(st + (size_t)rt * 16 * 256 + col + kb * 4) = tot[rt][c];
      }
    }
    return;
  }
  // ---- epilogue: lane (kb, ni) holds row rt * 16 + ni, columns kb * 4 .. + 3 of column tile c.  Through buffer accesses whose bounds drop what
  // lies past M and N: no branch per element, the exponentials and divisions of neighbours overlap (with a branch around every
  // element they ran one after the other: the epilogue was 15 % of the gate / up pair's time) ----
  const int rows = min(BM, a.M - m0);
  const bool wide = a.wide_out != 0;   // (uniform) four columns of a row are one aligned access
  constexpr int OB = EPI == EPI_ADDTO ? 4 : 2;
  const int ldo = EPI == EPI_ADDTO ? a.N : a.ldy;
  const auto view = [&](const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(p) + (size_t)m0 * ldo * OB), 0, p ? ((rows - 1) * ldo + a.N) * OB : 0, 0x00020000);
  };
  const auto out = view(EPI == EPI_ADDTO ? a.h_out : a.y);
  const auto res = view(EPI == EPI_ADDTO ? static_cast<const void*>(a.h_res) : EPI == EPI_STD ? a.residual : nullptr);
#pragma unroll
  for (int c = 0; c < (DUAL ? HCW : PF_CW); ++c) {
    const int n = tile[c] * 16 + kb * 4;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (EPI == EPI_STD) {
      if (a.bias) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[r] = load_ft<FT>(a.bias, min(n + r, a.N - 1));
      }
    }
    // byte offset of an element; what may not be touched lies outside every view
    const auto at = [&](int rt, int r) {
      const int row = (wm * PF_RT + rt) * 16 + ni;
      return tile_ok[c] && n + r < a.N && row < rows ? (row * ldo + n + r) * OB : 0x7FFFFFF0;
    };
#pragma unroll
    for (int rt = 0; rt < PF_RT; ++rt) {
      f32x4_t v = tot[rt][c];
      if constexpr (DUAL) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (v[r] / (1.f + expf(-v[r]))) * tot[rt][HCW + c][r];
      } else if constexpr (EPI == EPI_STD) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = a.alpha * v[r];
          if (a.bias) v[r] += bias[r];
          v[r] = apply_act(v[r], a.act);
        }
        if (a.residual) {
          u32x2_t q;
          if (wide) {
            q = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(res, at(rt, 0), 0, 0));
          } else {
            uint32_t e[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) e[r] = __builtin_amdgcn_raw_buffer_load_b16(res, at(rt, r), 0, 0);
            q = u32x2_t{e[0] | e[1] << 16, e[2] | e[3] << 16};
          }
          const u32x2_t w = {pack_ft2<FT>(v[0], v[1]), pack_ft2<FT>(v[2], v[3])};
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = ft_bits_to_f32<FT>((w[r >> 1] >> (r & 1) * 16) & 0xFFFFu) + ft_bits_to_f32<FT>((q[r >> 1] >> (r & 1) * 16) & 0xFFFFu);
        }
      } else {
        f32x4_t base;   // (no h_res: an empty view, zeros)
        if (wide) {
          base = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(res, at(rt, 0), 0, 0));
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) base[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(res, at(rt, r), 0, 0));
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = base[r] + a.alpha * v[r];
      }
      if constexpr (EPI == EPI_ADDTO) {
        if (wide) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), out, at(rt, 0), 0, 0);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v[r]), out, at(rt, r), 0, 0);
        }
      } else {
        const u32x2_t q = {pack_ft2<FT>(v[0], v[1]), pack_ft2<FT>(v[2], v[3])};
        if (wide) {
          __builtin_amdgcn_raw_buffer_store_b64(q, out, at(rt, 0), 0, 0);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(q[r >> 1] >> (r & 1) * 16), out, at(rt, r), 0, 0);
        }
      }
    }
  }
}

// split in K: the K parts of every split tile added in order + the epilogue of gemm_prefill_kernel.  4 columns per thread: bound by the slab's
// bytes (one column per thread took 14.7 us for 9 parts of 217 x 3584, 2.0 TB/s).
template <int FT, int EPI>
__global__ __launch_bounds__(256) void gemm_prefill_tail_reduce_kernel(const PrefillArgs a) {
  constexpr bool DUAL = EPI == EPI_SWIGLU;
  constexpr int NC = DUAL ? 128 : 256;  // output columns of a workgroup tile
  const int pitch = a.bm * 256;
  const int mblocks = (a.M + a.bm - 1) / a.bm;
  const size_t total = (size_t)(a.col_blocks - a.tail_cb) * a.M * (NC / 4);
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const int col = (int)(e % (NC / 4)) * 4;
    const size_t q = e / (NC / 4);
    const int cbt = (int)(q / a.M), m = (int)(q - (size_t)cbt * a.M), mb = m / a.bm, row = m - mb * a.bm;
    const int n0 = (a.tail_cb + cbt) * NC + col;
    if (n0 >= a.N) continue;
    const float* st = a.slab + (size_t)(cbt * mblocks + mb) * a.ksplit * pitch + (size_t)row * 256 + col;
    f32x4_t v4 = {0.f, 0.f, 0.f, 0.f}, u4 = v4;
    for (int s = 0; s < a.ksplit; ++s) {
      v4 += *reinterpret_cast<const f32x4_t*>(st + (size_t)s * pitch);
      if constexpr (DUAL) u4 += *reinterpret_cast<const f32x4_t*>(st + (size_t)s * pitch + 128);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + r;
      if (n >= a.N) break;
      float v = v4[r];
      if constexpr (DUAL) {
        store_ft<FT>(a.y, (size_t)m * a.ldy + n, (v / (1.f + expf(-v))) * u4[r]);
      } else if constexpr (EPI == EPI_STD) {
        v = a.alpha * v;
        if (a.bias) v += load_ft<FT>(a.bias, n);
        v = apply_act(v, a.act);
        if (a.residual) v = ft_round<FT>(v) + load_ft<FT>(a.residual, (size_t)m * a.ldy + n);
        store_ft<FT>(a.y, (size_t)m * a.ldy + n, v);
      } else {
        const float base = a.h_res ? a.h_res[(size_t)m * a.N + n] : 0.f;
        a.h_out[(size_t)m * a.N + n] = base + a.alpha * v;
      }
    }
  }
}

template <int WBITS, int FT, int EPI, int GPT>
hipError_t launch_gemm_prefill(const PrefillArgs& a, int blocks, hipStream_t stream);

template <int WBITS, int FT, int EPI, int GPT, int TR, int UK>
hipError_t launch_gemm_prefill_unit(const PrefillArgs& a, int blocks, hipStream_t s) {
  auto kern = gemm_prefill_kernel<WBITS, FT, EPI, GPT, TR, UK>;
  constexpr size_t lds = prefill_lds_bytes<WBITS, TR, UK>();
  if (lds > 64 * 1024) {  // the grant is per device: once per device of this process
    static std::atomic<unsigned> granted_mask[4];  // 128 device ids
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipGetLastError();
    const unsigned bit = 1u << (dev & 31);
    std::atomic<unsigned>* word = dev >= 0 && dev < 128 ? &granted_mask[dev >> 5] : nullptr;
    if (!word || !(word->load(std::memory_order_acquire) & bit)) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
      if (word) word->fetch_or(bit, std::memory_order_release);
    }
  }
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(PF_THREADS), lds, s, a);
  if (a.tail_cb < a.col_blocks) {
    const size_t quads = (size_t)(a.col_blocks - a.tail_cb) * a.M * (EPI == EPI_SWIGLU ? 32 : 64);
    hipLaunchKernelGGL((gemm_prefill_tail_reduce_kernel<FT, EPI>), dim3((unsigned)std::min<size_t>((quads + 255) / 256, 4096)), dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

// (a group of an odd number of k-tiles ends between two of them)
template <int WBITS, int FT, int EPI, int GPT, int TR>
hipError_t launch_gemm_prefill_rows(const PrefillArgs& a, int blocks, hipStream_t s) {
  if constexpr (WBITS == 8 && !GPT) {
    if (a.ktpg % 2 == 0) return launch_gemm_prefill_unit<WBITS, FT, EPI, GPT, TR, 2>(a, blocks, s);
  }
  return launch_gemm_prefill_unit<WBITS, FT, EPI, GPT, TR, 1>(a, blocks, s);
}

#define DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI, GPT)                                                                \
  template <>                                                                                                           \
  hipError_t launch_gemm_prefill<WBITS, FT, EPI, GPT>(const PrefillArgs& a, int blocks, hipStream_t s) {                \
    switch (a.bm / 16) {                                                                                                \
      case 5: return launch_gemm_prefill_rows<WBITS, FT, EPI, GPT, 5>(a, blocks, s);                                    \
      case 6: return launch_gemm_prefill_rows<WBITS, FT, EPI, GPT, 6>(a, blocks, s);                                    \
      case 7: return launch_gemm_prefill_rows<WBITS, FT, EPI, GPT, 7>(a, blocks, s);                                    \
      default: return launch_gemm_prefill_rows<WBITS, FT, EPI, GPT, 8>(a, blocks, s);                                   \
    }                                                                                                                   \
  }

#define DIHIP_DEFINE_PREFILL_LAUNCH_SET(WBITS, FT)          \
  DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI_STD, 0)        \
  DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI_STD, 1)        \
  DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI_SWIGLU, 0)     \
  DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI_SWIGLU, 1)     \
  DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI_ADDTO, 0)      \
  DIHIP_DEFINE_PREFILL_LAUNCH(WBITS, FT, EPI_ADDTO, 1)

}  // namespace dihip
