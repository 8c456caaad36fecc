// seq_gla_gated.hip -- gated linear attention from the rows of its input product to the rows of its output product, in one kernel (three for long portions):
//   z = bf16(a1 h) . a2^T + b2 (matrix cores, f32 sums),   alpha = sigmoid(z)^(1/tau),   S <- diag(alpha) S + k v^T,   o = S^T (q * q_scale),
//   y[t, h, :] = o / rms(o) * gamma * gate[t, h, :]
// The state, its decays, keys, values, queries and sums are f32.  The arithmetic of the recurrence and of the norm is that of seq_gla.hip, which serves every other size
// and type; long portions run as chunks side by side as they do there.
//
// A workgroup owns one head: its 4 waves hold a quarter of the channels of S each, a lane two columns (lane, lane + 64).  What bounds it is the chain over the rows of a chunk: seq_gla.hip
// fetched a row's decays, keys and queries by scalar loads, which wait for the L2 at every row (about 2000 clocks of a row for 400 of arithmetic).  Here 16 rows at a time
// are staged in LDS while the 16 before are multiplied: 16 rows x 16 channels of z are one or a few MFMAs per wave, then a row costs 16-byte broadcast reads.
// The rows' outputs meet in LDS anyway, so the norm over a head and the gate are applied there: the separate launches for z, the rows' records and the norm go, and
// with them their f32 rows in memory.
// All launches from z to the norm, us, before -> this: 500 rows beside 13 portions of one (16 heads of 64 x 128, rank 64) 162 -> 45; 2048 rows (32 heads) 252 -> 150, of which the
// recurrence's multiply-adds, three per row, channel and column and two in PASS 1, are 80; 24 portions of one 27.3 -> 11.2 (25 MB of state out and in); one 25.4 -> 7.0.
#include <algorithm>
#include "seq_common.h"
#include "seq_linear.h"

namespace dihip {
namespace {

constexpr int GG_RB = 16, GG_SUB = 8;   // rows staged at a time; rows between two exchanges of partial sums

// floats of a staged row: decay, key, scaled query of 4 * dpt channels; padded so that 16 rows' pieces fall on different banks, unless that would cost the second workgroup of a CU
constexpr int gg_row(int dpt) { return 12 * dpt + (dpt == 16 ? 4 : 0); }

struct GlaGatedArgs {
  void* y; int ydt; long ldy;
  const float* q; const float* k; const float* v; const float* gate; const float* a1; long ld;   // columns of the same rows
  const uint16_t* a2; const uint16_t* b2; const uint16_t* gamma;                                 // bf16
  float q_scale, inv_tau, eps;
  float* state;
  const int32_t* ent_slot; const int32_t* ent_row0; const int32_t* ent_count;
  int E, H, D, DV, chunk, chunks;   // (chunks: records there are)
  float* ws;   // [chunk in gg_chunk's order][H] records: D * DV (state) + D (product of the decays) floats
};

// log(1 + x), 0 <= x <= 1: 2 atanh(x / (2 + x)), whose argument is at most a third: eight terms of the series (s .. s^15 / 15) leave 1.5e-9 of it.  (log1pf keeps a sum in two floats: 75 instructions,
// a third of the recurrence's own.)
__device__ __forceinline__ float gg_log1p(float x) {
  const float d = 2.f + x, r = __builtin_amdgcn_rcpf(d), s0 = x * r;
  const float s = __builtin_fmaf(__builtin_fmaf(-d, s0, x), r, s0), w = s * s;
  float p = 1.f / 15;
  p = __builtin_fmaf(p, w, 1.f / 13);
  p = __builtin_fmaf(p, w, 1.f / 11);
  p = __builtin_fmaf(p, w, 1.f / 9);
  p = __builtin_fmaf(p, w, 1.f / 7);
  p = __builtin_fmaf(p, w, 1.f / 5);
  p = __builtin_fmaf(p, w, 1.f / 3);
  return 2.f * __builtin_fmaf(p * w, s, s);
}
__device__ __forceinline__ float gg_log_sigmoid(float z) { return -(gg_log1p(expf(-fabsf(z))) + fmaxf(-z, 0.f)); }

// the portion and chunk of workgroup b among all chunks of all portions, portion by portion; false: there are fewer.  (A grid over the longest portion's chunks is mostly
// workgroups that wait for LDS to find nothing: 500 rows beside 13 portions of one, 64 us with them.)
__device__ __forceinline__ bool gg_chunk(const int32_t* __restrict__ count, int E, int chunk, int b, int& e, int& ch) {
  const int lane = threadIdx.x & 63;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int mine = e0 + lane < E ? (max(count[e0 + lane], 0) + chunk - 1) / chunk : 0;
    int upto = mine;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const int other = __shfl_up(upto, d, 64);
      if (lane >= d) upto += other;
    }
    const uint64_t past = __builtin_amdgcn_ballot_w64(upto > b);
    if (past) {
      const int l = __builtin_ctzll(past);
      e = e0 + l;
      ch = b - (__builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(mine, l));
      return true;
    }
    b -= __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// the number of portion e's first chunk in that order (every lane of the wave)
__device__ __forceinline__ int gg_first(const int32_t* __restrict__ count, int e, int chunk) {
  const int lane = threadIdx.x & 63;
  int n = 0;
  for (int i = lane; i < e; i += 64) n += (max(count[i], 0) + chunk - 1) / chunk;
#pragma unroll
  for (int d = 32; d > 0; d /= 2) n += __shfl_xor(n, d, 64);
  return n;
}

// PASS 0: whole portions from the slot's state.  PASS 1: every chunk but the last from S = 0 -> its record.  PASS 3: every chunk from the state that the carry left in its record
// (portions of one chunk: from the slot's).  RS: 32-element steps of the rank.
template <int DPT, int RS, int PASS>
__global__ __launch_bounds__(256, 2) void gla_gated_kernel(GlaGatedArgs a) {
  constexpr int DP = 4 * DPT, LDR = gg_row(DPT), TILES = DP / 64, QUADS = DP / 64;   // 16-channel tiles of z per wave; 4-channel units of a staged row per thread
  constexpr bool OUT = PASS != 1;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* rec = lds;                                   // [2][GG_RB][LDR]
  float* part = lds + 2 * GG_RB * LDR;                // [GG_SUB][4][128] (not PASS 1)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int D = a.D, DV = a.DV, h = blockIdx.y;
  int e = blockIdx.x, ch = 0;
  if (PASS != 0 && !gg_chunk(a.ent_count, a.E, a.chunk, blockIdx.x, e, ch)) return;
  const int cnt = __builtin_amdgcn_readfirstlane(a.ent_count[e]);
  const int lo = PASS == 0 ? 0 : ch * a.chunk;
  const int first_row = __builtin_amdgcn_readfirstlane(a.ent_row0[e]), slot = __builtin_amdgcn_readfirstlane(a.ent_slot[e]);
  if (lo >= cnt || (PASS == 1 && lo + a.chunk >= cnt)) return;
  const int n = PASS == 0 ? cnt : min(a.chunk, cnt - lo);
  const size_t row0 = (size_t)first_row + lo;
  float* wrec = PASS == 0 ? nullptr : a.ws + ((size_t)blockIdx.x * a.H + h) * ((size_t)D * DV + D);
  float* sp = a.state + ((size_t)slot * a.H + h) * D * DV;
  // columns past the head and rows past the end are loaded from the last one: loads under a condition each would be a branch each
  const bool col[2] = {lane < DV, lane + 64 < DV};
  const int cj[2] = {min(lane, DV - 1), min(lane + 64, DV - 1)};
  const int c0 = wave * DPT;   // the wave's first channel
  float S[DPT][2];
  {
    const float* from = PASS == 0 || cnt <= a.chunk ? sp : wrec;
#pragma unroll
    for (int i = 0; i < DPT; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c) S[i][c] = PASS == 1 ? 0.f : from[min(c0 + i, D - 1) * DV + cj[c]];
  }
  // staging: fetch() asks for the rows b0 .. b0 + 15, put() leaves their records in LDS.  Rows past the end keep the state: decay 1, key 0
  u32x4_t wz[TILES][RS];
  f32x4_t bz[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const int ch0 = (wave + 4 * t) * 16;
    if (ch0 >= D) continue;
    const size_t first = (size_t)h * D + ch0;
#pragma unroll
    for (int s = 0; s < RS; ++s) wz[t][s] = *reinterpret_cast<const u32x4_t*>(a.a2 + (first + (lane & 15)) * (RS * 32) + s * 32 + (lane >> 4) * 8);
    const u32x2_t u = *reinterpret_cast<const u32x2_t*>(a.b2 + first + (lane >> 4) * 4);
    bz[t] = f32x4_t{bf16_bits_to_f32(u[0] & 0xffffu), bf16_bits_to_f32(u[0] >> 16), bf16_bits_to_f32(u[1] & 0xffffu), bf16_bits_to_f32(u[1] >> 16)};
  }
  f32x4_t fx[RS][2], fk[QUADS], fq[QUADS];
  auto fetch = [&](int b0) {
    const float* xr = a.a1 + (row0 + min(b0 + (lane & 15), n - 1)) * a.ld + (lane >> 4) * 8;
#pragma unroll
    for (int s = 0; s < RS; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i) fx[s][i] = *reinterpret_cast<const f32x4_t*>(xr + s * 32 + i * 4);
#pragma unroll
    for (int u = 0; u < QUADS; ++u) {
      const int r = (tid + 256 * u) / (DP / 4), c = (tid + 256 * u) % (DP / 4) * 4;
      const size_t at = (row0 + min(b0 + r, n - 1)) * a.ld + (size_t)h * D + min(c, D - 4);
      fk[u] = *reinterpret_cast<const f32x4_t*>(a.k + at);
      if (OUT) fq[u] = *reinterpret_cast<const f32x4_t*>(a.q + at);
    }
  };
  auto put = [&](int b0, float* to) {
    u32x4_t x[RS];
#pragma unroll
    for (int s = 0; s < RS; ++s)
      x[s] = u32x4_t{pack_bf16x2(fx[s][0][0], fx[s][0][1]), pack_bf16x2(fx[s][0][2], fx[s][0][3]), pack_bf16x2(fx[s][1][0], fx[s][1][1]), pack_bf16x2(fx[s][1][2], fx[s][1][3])};
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int ch0 = (wave + 4 * t) * 16;
      f32x4_t al = {1.f, 1.f, 1.f, 1.f};
      if (ch0 < D) {
        f32x4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < RS; ++s) z = mfma_bf16(wz[t][s], x[s], z);
        z += bz[t];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = expf(gg_log_sigmoid(z[i]) * a.inv_tau);
          al[i] = b0 + (lane & 15) < n ? v : 1.f;
        }
      }
      *reinterpret_cast<f32x4_t*>(to + (lane & 15) * LDR + ch0 + (lane >> 4) * 4) = al;
    }
#pragma unroll
    for (int u = 0; u < QUADS; ++u) {
      const int r = (tid + 256 * u) / (DP / 4), c = (tid + 256 * u) % (DP / 4) * 4;
      const bool in = b0 + r < n && c < D;
      float* p = to + r * LDR + c;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        fk[u][i] = in ? fk[u][i] : 0.f;
        if (OUT) fq[u][i] = in ? fq[u][i] * a.q_scale : 0.f;
      }
      *reinterpret_cast<f32x4_t*>(p + DP) = fk[u];
      if (OUT) *reinterpret_cast<f32x4_t*>(p + 2 * DP) = fq[u];
    }
  };
  float vr[GG_SUB][2];
  const float* vhead = a.v + row0 * a.ld + (size_t)h * DV;
  const float* ghead = a.gate + row0 * a.ld + (size_t)h * DV;
  auto fetch_v = [&](int b0) {
#pragma unroll
    for (int r = 0; r < GG_SUB; ++r) {
      const float* vp = vhead + (size_t)min(b0 + r, n - 1) * a.ld;
#pragma unroll
      for (int c = 0; c < 2; ++c) vr[r][c] = vp[cj[c]];
    }
  };
  float gam[2] = {0.f, 0.f};
  if (OUT) {
#pragma unroll
    for (int c = 0; c < 2; ++c) gam[c] = bf16_bits_to_f32(a.gamma[cj[c]]);
  }
  float ap = 1.f;   // PASS 1: the product of the decays of channel c0 + lane % DPT
  fetch(0);
  fetch_v(0);
  put(0, rec);
  __syncthreads();
  for (int b0 = 0; b0 < n; b0 += GG_RB) {
    const float* here = rec + (b0 / GG_RB & 1) * (GG_RB * LDR);
    float* next = rec + (~(b0 / GG_RB) & 1) * (GG_RB * LDR);
    const bool more = b0 + GG_RB < n;   // (uniform, as everything that decides about a barrier)
    if (more) fetch(b0 + GG_RB);
#pragma unroll
    for (int sub = 0; sub < GG_RB / GG_SUB; ++sub) {
      const int s0 = b0 + sub * GG_SUB;
      const bool live = s0 < n;
      float vc[GG_SUB][2], gt[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll
      for (int r = 0; r < GG_SUB; ++r)
#pragma unroll
        for (int c = 0; c < 2; ++c) vc[r][c] = s0 + r < n ? vr[r][c] : 0.f;   // (a row past the end has key 0, but an infinity times 0 is none)
      if (s0 + GG_SUB < n) fetch_v(s0 + GG_SUB);
      if (OUT && live) {   // the gates of the rows that this wave will finish
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float* gp = ghead + (size_t)min(s0 + wave * 2 + r, n - 1) * a.ld;
#pragma unroll
          for (int c = 0; c < 2; ++c) gt[r][c] = gp[cj[c]];
        }
      }
#pragma unroll
      for (int r0 = 0; r0 < GG_SUB; r0 += 4) {
        if (s0 + r0 < n) {
#pragma unroll
          for (int r = r0; r < r0 + 4; ++r) {
            const float* rr = here + (sub * GG_SUB + r) * LDR + c0;
            float po[2] = {0.f, 0.f};
#pragma unroll
            for (int i0 = 0; i0 < DPT; i0 += 4) {
              const f32x4_t a4 = *reinterpret_cast<const f32x4_t*>(rr + i0), k4 = *reinterpret_cast<const f32x4_t*>(rr + DP + i0);
              f32x4_t q4 = {0.f, 0.f, 0.f, 0.f};
              if (OUT) q4 = *reinterpret_cast<const f32x4_t*>(rr + 2 * DP + i0);
#pragma unroll
              for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                  S[i0 + i][c] = __builtin_fmaf(a4[i], S[i0 + i][c], k4[i] * vc[r][c]);
                  if (OUT) po[c] = __builtin_fmaf(S[i0 + i][c], q4[i], po[c]);
                }
            }
            if (PASS == 1) ap *= rr[lane % DPT];
            if (OUT) {
#pragma unroll
              for (int c = 0; c < 2; ++c) part[(r * 4 + wave) * 128 + lane + 64 * c] = po[c];
            }
          }
        }
      }
      if (sub == GG_RB / GG_SUB - 1 && more) put(b0 + GG_RB, next);
      if (OUT || sub == GG_RB / GG_SUB - 1) __syncthreads();
      if (OUT && live) {
#pragma unroll
        for (int rw = 0; rw < 2; ++rw) {
          const int r = wave * 2 + rw;
          if (s0 + r >= n) continue;
          float o[2], ss = 0.f;
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const float* p = part + r * 4 * 128 + lane + 64 * c;
            o[c] = (p[0] + p[128]) + (p[256] + p[384]);
            if (col[c]) ss = __builtin_fmaf(o[c], o[c], ss);
          }
          const float inv = 1.f / sqrtf(wave_sum(ss) / (float)DV + a.eps);
#pragma unroll
          for (int c = 0; c < 2; ++c)
            if (col[c]) st_any(a.y, (row0 + s0 + r) * a.ldy + (size_t)h * DV + lane + 64 * c, a.ydt, o[c] * inv * gam[c] * gt[rw][c]);
        }
      }
      if (OUT && s0 + GG_SUB < n) __syncthreads();   // part has been read
    }
  }
  if (PASS != 3 || lo + n == cnt) {
    float* dst = PASS == 1 ? wrec : sp;
#pragma unroll
    for (int i = 0; i < DPT; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        if (c0 + i < D && col[c]) dst[(size_t)(c0 + i) * DV + lane + 64 * c] = S[i][c];
    if (PASS == 1 && lane < DPT && c0 + lane < D) wrec[(size_t)D * DV + c0 + lane] = ap;
  }
}

// chunks in order, 4 state elements per thread: record <- the state its chunk starts from;  S <- decay product * S + record
__global__ __launch_bounds__(256) void gla_gated_carry_kernel(GlaGatedArgs a) {
  const int e = blockIdx.z, h = blockIdx.y, idx = (blockIdx.x * 256 + threadIdx.x) * 4;
  const int chunks = (a.ent_count[e] + a.chunk - 1) / a.chunk;
  if (chunks < 2) return;   // (uniform)
  const int first = gg_first(a.ent_count, e, a.chunk);
  if (idx >= a.D * a.DV || first + chunks > a.chunks) return;
  const size_t size = (size_t)a.D * a.DV + a.D, step = (size_t)a.H * size;
  float* w0 = a.ws + ((size_t)first * a.H + h) * size;
  const int i = idx / a.DV;   // (DV % 4 == 0: one channel)
  f32x4_t S = *reinterpret_cast<const f32x4_t*>(a.state + ((size_t)a.ent_slot[e] * a.H + h) * a.D * a.DV + idx);
  constexpr int U8 = 8;       // eight chunks' records in flight
  for (int c0 = 0; c0 < chunks; c0 += U8) {
    f32x4_t U[U8];
    float A[U8];
#pragma unroll
    for (int x = 0; x < U8; ++x) {   // (the last chunk has no record yet, and needs none)
      const int ch = min(c0 + x, chunks - 2);
      U[x] = *reinterpret_cast<const f32x4_t*>(w0 + ch * step + idx);
      A[x] = w0[ch * step + (size_t)a.D * a.DV + i];
    }
#pragma unroll
    for (int x = 0; x < U8; ++x) {
      if (c0 + x < chunks) {
        *reinterpret_cast<f32x4_t*>(w0 + (c0 + x) * step + idx) = S;
#pragma unroll
        for (int j = 0; j < 4; ++j) S[j] = __builtin_fmaf(A[x], S[j], U[x][j]);
      }
    }
  }
}

bool gla_gated_fits(int H, int D, int DV, int rank) {
  return H > 0 && H <= 65535 && D > 0 && D <= 128 && D % 16 == 0 && DV > 0 && DV <= 128 && DV % 4 == 0 && rank > 0 && rank <= 128 && rank % 32 == 0;
}
// rows of a chunk: as many workgroups as 256 CUs hold two of, if the portions have the rows; a chunk costs a state out and in again, so short ones only where few rows leave CUs idle
int gla_gated_chunk(int max_count, int H) {
  for (int rows = 64; rows > 16; rows /= 2)
    if ((long)((max_count + rows - 1) / rows) * H >= 512) return rows;
  return max_count > 128 ? 32 : 16;
}

// no more chunks than these, however the T rows are cut into E portions of at most max_count: a record each (numbered portion by portion.  With room for max_count rows in
// every portion, 700 rows beside 24 of one and 32 heads took 581 MB for the 46 chunks that there are; 47 records are 50 MB)
long gla_gated_chunks(int T, int E, int max_count, int rows) { return std::min<long>((long)E * ((max_count + rows - 1) / rows), T / rows + (long)E); }

}  // namespace
}  // namespace dihip

using namespace dihip;

extern "C" {

int dihip_gla_gated_supported(int H, int D, int DV, int rank) { return gla_gated_fits(H, D, DV, rank) ? 1 : 0; }

size_t dihip_gla_gated_workspace_bytes(int T, int E, int max_count, int H, int D, int DV) {
  if (T <= 0 || E <= 0 || H <= 0 || D <= 0 || DV <= 0 || max_count <= 16) return 0;
  const int rows = gla_gated_chunk(max_count, H);
  return (size_t)gla_gated_chunks(T, E, max_count, rows) * H * ((size_t)D * DV + D) * sizeof(float);
}

int dihip_gla_gated(void* stream, void* y, int y_dtype, long ldy, const float* q, const float* k, const float* v, const float* gate, const float* a1, long ld,
                    const void* a2, const void* a2_bias, const void* gamma, int rank, float q_scale, float tau, float eps, float* state, const int32_t* ent_slot,
                    const int32_t* ent_row0, const int32_t* ent_count, int T, int E, int max_count, int H, int D, int DV, void* ws, size_t ws_bytes) {
  DIHIP_REQUIRE(T >= 0 && E >= 0 && max_count >= 0 && y && q && k && v && gate && a1 && a2 && a2_bias && gamma && state && ent_slot && ent_row0 && ent_count &&
                    seq_dtype_ok(y_dtype) && tau > 0.f, DIHIP_PARAM_ERROR, "gla_gated: bad argument");
  DIHIP_REQUIRE(gla_gated_fits(H, D, DV, rank), DIHIP_EXCEED_LIMIT_ERROR, "gla_gated: D %d DV %d rank %d", D, DV, rank);
  DIHIP_REQUIRE(ldy >= (long)H * DV && ld >= (long)H * D && ld >= (long)H * DV && ld >= rank && E <= 65535, DIHIP_PARAM_ERROR, "gla_gated: bad argument");
  DIHIP_REQUIRE(ld % 4 == 0 && ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(a1) | reinterpret_cast<uintptr_t>(a2) |
                                 reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(ws)) & 15u) == 0 && (reinterpret_cast<uintptr_t>(a2_bias) & 7u) == 0,
                DIHIP_PARAM_ERROR, "gla_gated: queries, keys, a1, a2, state and workspace start on 16 bytes, and so does every row");
  if (T == 0 || E == 0 || max_count == 0) return DIHIP_SUCCESS;
  const bool chunked = max_count > 16;
  DIHIP_REQUIRE(!chunked || (ws && ws_bytes >= dihip_gla_gated_workspace_bytes(T, E, max_count, H, D, DV)), DIHIP_PARAM_ERROR, "gla_gated: workspace too small");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int rows = chunked ? gla_gated_chunk(max_count, H) : max_count, all = (int)gla_gated_chunks(T, E, max_count, rows);
  const GlaGatedArgs a{y, y_dtype, ldy, q, k, v, gate, a1, ld, (const uint16_t*)a2, (const uint16_t*)a2_bias, (const uint16_t*)gamma, q_scale, 1.f / tau, eps, state,
                       ent_slot, ent_row0, ent_count, E, H, D, DV, rows, all, (float*)ws};
  auto go = [&](auto dpt, auto rs) {
    constexpr int DPT = decltype(dpt)::value, RS = decltype(rs)::value, REC = 2 * GG_RB * gg_row(DPT) * 4, PART = GG_SUB * 4 * 128 * 4;
    static_assert(REC + PART <= 65536, "what a launch may ask for without a grant");
    if (!chunked) {
      hipLaunchKernelGGL((gla_gated_kernel<DPT, RS, 0>), dim3(E, H), dim3(256), REC + PART, s, a);
      return;
    }
    hipLaunchKernelGGL((gla_gated_kernel<DPT, RS, 1>), dim3(all, H), dim3(256), REC, s, a);
    hipLaunchKernelGGL(gla_gated_carry_kernel, dim3((D * DV / 4 + 255) / 256, H, E), dim3(256), 0, s, a);
    hipLaunchKernelGGL((gla_gated_kernel<DPT, RS, 3>), dim3(all, H), dim3(256), REC + PART, s, a);
  };
  auto by_rank = [&](auto dpt) {
    switch (rank / 32) {
      case 1: return go(dpt, std::integral_constant<int, 1>{});
      case 2: return go(dpt, std::integral_constant<int, 2>{});
      case 3: return go(dpt, std::integral_constant<int, 3>{});
      default: return go(dpt, std::integral_constant<int, 4>{});
    }
  };
  if (D <= 64) by_rank(std::integral_constant<int, 16>{});
  else by_rank(std::integral_constant<int, 32>{});
  return launch_status();
}

}  // extern "C"
