// seq_gqa.hip -- grouped-query attention over paged key and value caches for the sequence engine:
//   qkv_prep_append   per token: unit-RMS norm of every query / key head (optional), rotary positions (paired or half-split
//                     layout, a frequency table and a magnitude from the host), mixing of the values with another layer's,
//                     queries written back in place, keys and values appended to their pages
//   qkv_conv_prep_append   the same for a layer with a short causal convolution on every channel of q, k and v and norms over the
//                     whole query / key row
//   gqa_attn_kernel   one workgroup per row, every product and sum in f32 (any cache type)
//   gqa_attn_mc_kernel + merge   bf16 caches on the matrix cores, the key walk split for few rows (decoding)
// Options of the softmax: a sink logit per head or the constant 0 (one more term in the denominator, no value), a tanh cap on
// the scores, a multiplier per (row, head) on the output (the output gate).
// Options of the key walk: a sliding window with kept first keys (row p reads key j <= p if p - j < window or j < keep_first;
// the keys between are skipped by whole chunks / tiles), and several softmax maps per head (`maps`: head h has maps query
// vectors and its key head maps key vectors, laid out one after the other; map m of a head scores against map m of its key
// head, all maps read the same values; the output holds the maps of a head side by side).
//   maps_diff_norm    two maps per head -> one: (first - lam * second) / its root mean square * a constant
#include "seq_common.h"

namespace dihip {
namespace {

// ------------------------------------------------------------------------------------------------ prep + append
struct PrepArgs {
  float* qkv; long ld; int q_off, k_off, v_off;
  int H, G, D, DV, GV;   // H / G: query / key vectors per token (heads x maps), GV: value heads
  const void* qnorm; const void* knorm; int wdt; float eps;
  const float* freq; int rot_dims, layout; float mag;
  float lam; const float* vfirst_in; float* vfirst_out; long ldvf;
  void* const* kspans; void* const* vspans; int span_stride, span_len, cdt;
  const int32_t* tok_slot; const int32_t* tok_pos;
};

__global__ __launch_bounds__(256) void qkv_prep_append_kernel(PrepArgs a) {
  __shared__ float hs[4][256];
  __shared__ float cs_t[128], sn_t[128];   // the token's cos and sin per rotated pair, shared by all heads
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pos = a.tok_pos[t];
  if (threadIdx.x < (a.rot_dims >> 1)) {
    float sn, cs;
    rope_sincos((uint32_t)pos, a.freq[threadIdx.x], &sn, &cs);
    cs_t[threadIdx.x] = cs * a.mag;
    sn_t[threadIdx.x] = sn * a.mag;
  }
  const size_t sp = (size_t)a.tok_slot[t] * a.span_stride + pos / a.span_len;
  const size_t in_span = (size_t)(pos % a.span_len);
  float* row = a.qkv + (size_t)t * a.ld;
  const int D = a.D, half = a.rot_dims >> 1;
  for (int h0 = blockIdx.y * 4; h0 < a.H + a.G; h0 += 4 * gridDim.y) {      // query heads, then key heads: the same trip count in every wave
    const int hh = h0 + wave;
    const bool live = hh < a.H + a.G, is_q = hh < a.H;
    float* src = row + (is_q ? a.q_off + hh * D : a.k_off + (hh - a.H) * D);
    const void* gamma = is_q ? a.qnorm : a.knorm;
    float v[4], ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = lane + 64 * i;
      v[i] = live && d < D ? src[d] : 0.f;
      ss = __builtin_fmaf(v[i], v[i], ss);
    }
    if (gamma) {
      const float inv = 1.f / sqrtf(wave_sum(ss) / (float)D + a.eps);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = lane + 64 * i;
        if (d < D) v[i] = v[i] * inv * ld_any(gamma, d, a.wdt);
      }
    }
    __syncthreads();   // hs of the head before is no longer read
#pragma unroll
    for (int i = 0; i < 4; ++i) hs[wave][lane + 64 * i] = v[i];
    __syncthreads();
    if (live) {
      void* kdst = is_q ? nullptr : a.kspans[sp];
      const size_t kbase = (in_span * a.G + (size_t)(is_q ? 0 : hh - a.H)) * D;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = lane + 64 * i;
        if (d >= D) continue;
        float y = v[i];
        if (d < a.rot_dims) {
          int pair, other;
          bool first;
          if (a.layout == 0) { pair = d >> 1; first = (d & 1) == 0; other = d ^ 1; }
          else { first = d < half; pair = first ? d : d - half; other = first ? d + half : d - half; }
          const float sn = sn_t[pair], cs = cs_t[pair];
          const float o = hs[wave][other];
          y = first ? v[i] * cs - o * sn : v[i] * cs + o * sn;
        }
        if (is_q) src[d] = y;
        else st_any(kdst, kbase + d, a.cdt, y);
      }
    }
  }
  void* vdst = a.vspans[sp];
  const int nv = a.GV * a.DV;
  for (int e = blockIdx.y * 256 + threadIdx.x; e < nv; e += 256 * gridDim.y) {
    float v = row[a.v_off + e];
    if (a.vfirst_in) v = (1.f - a.lam) * v + a.lam * a.vfirst_in[(size_t)t * a.ldvf + e];
    if (a.vfirst_out) a.vfirst_out[(size_t)t * a.ldvf + e] = v;
    st_any(vdst, in_span * nv + e, a.cdt, v);
  }
}

// The same for head sizes of 64 and 128 in rows of whole 16-byte pieces and bf16 pages: a lane holds four neighbouring elements of a head, 16 or 32 lanes a head, every operand is
// read once and the heads of a wave are in flight together; no barrier after the token's table.  The kernel above, an element per lane and two barriers per four heads,
// waited for every group's loads.  Bound by the rows' bytes: 2048 rows of 32 + 8 heads of 128 40 -> 24 us (3.5 TB/s), 513 rows of 16 + 4 11.4 -> 7.7; decoding, one group of heads
// per wave, 4.9 and 5.0 (24 rows), 4.8 and 4.6 (one).
// PREP_HEADS: the groups of heads a wave has in flight
template <int D, int PREP_HEADS>
__global__ __launch_bounds__(256) void qkv_prep_append_vec_kernel(PrepArgs a) {
  constexpr int LPH = D / 4, HPW = 64 / LPH;   // lanes per head, heads per wave
  __shared__ float cs_t[64], sn_t[64];
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane % LPH, d0 = sub * 4;
  const int pos = a.tok_pos[t], nh = a.H + a.G, half = a.rot_dims >> 1;
  const size_t sp = (size_t)a.tok_slot[t] * a.span_stride + pos / a.span_len, in_span = (size_t)(pos % a.span_len);
  float* row = a.qkv + (size_t)t * a.ld;
  uint16_t* const kdst = (uint16_t*)a.kspans[sp];
  uint16_t* const vdst = (uint16_t*)a.vspans[sp];
  const int first = (blockIdx.y * 4 + wave) * HPW + lane / LPH, step = 4 * HPW * gridDim.y;
  auto column = [&](int h) { return h < a.H ? a.q_off + h * D : a.k_off + (h - a.H) * D; };
  f32x4_t v[PREP_HEADS];
  auto load = [&](int h0) {
#pragma unroll
    for (int i = 0; i < PREP_HEADS; ++i) {
      const int h = h0 + i * step;
      v[i] = *reinterpret_cast<const f32x4_t*>(row + column(min(h, nh - 1)) + d0);   // (past the heads: the last one's, not used)
    }
  };
  load(first);
  f32x4_t gq = {1.f, 1.f, 1.f, 1.f}, gk = gq;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (a.qnorm) gq[r] = ld_any(a.qnorm, d0 + r, a.wdt);
    if (a.knorm) gk[r] = ld_any(a.knorm, d0 + r, a.wdt);
  }
  if (threadIdx.x < half) {
    float sn, cs;
    rope_sincos((uint32_t)pos, a.freq[threadIdx.x], &sn, &cs);
    cs_t[threadIdx.x] = cs * a.mag;
    sn_t[threadIdx.x] = sn * a.mag;
  }
  __syncthreads();
  const bool turned = d0 < a.rot_dims, low = d0 < half;   // (rot_dims is a multiple of 8: a lane's four turn together)
  f32x4_t cs = {1.f, 1.f, 1.f, 1.f}, sn = {0.f, 0.f, 0.f, 0.f};
  if (turned) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pair = a.layout == 0 ? (d0 + r) >> 1 : low ? d0 + r : d0 + r - half;
      cs[r] = cs_t[pair];
      sn[r] = (a.layout == 0 ? (r & 1) == 0 : low) ? -sn_t[pair] : sn_t[pair];   // y = v cs +- other sn
    }
  }
  const int other = a.layout == 0 || !turned ? lane : low ? lane + half / 4 : lane - half / 4;
  const bool kwide = (reinterpret_cast<uintptr_t>(kdst) & 7) == 0, vwide = (reinterpret_cast<uintptr_t>(vdst) & 7) == 0;   // (uniform)
  auto store = [&](uint16_t* to, const f32x4_t& x, bool wide) {
    const uint32_t e[4] = {f32_to_bf16_bits(x[0]), f32_to_bf16_bits(x[1]), f32_to_bf16_bits(x[2]), f32_to_bf16_bits(x[3])};
    if (wide) *reinterpret_cast<u32x2_t*>(to) = u32x2_t{e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
    else
#pragma unroll
      for (int r = 0; r < 4; ++r) to[r] = (uint16_t)e[r];
  };
  for (int h0 = first, base = (int)blockIdx.y * 4 * HPW; base < nh; h0 += PREP_HEADS * step, base += PREP_HEADS * step) {   // (uniform)
    if (h0 != first) load(h0);
#pragma unroll
    for (int i = 0; i < PREP_HEADS; ++i) {
      const int h = h0 + i * step;
      const bool is_q = h < a.H;
      f32x4_t x = v[i];
      float ss = __builtin_fmaf(x[3], x[3], __builtin_fmaf(x[2], x[2], __builtin_fmaf(x[1], x[1], x[0] * x[0])));
#pragma unroll
      for (int m = 1; m < LPH; m *= 2) ss += __shfl_xor(ss, m, 64);
      if (is_q ? a.qnorm != nullptr : a.knorm != nullptr) {
        const float inv = 1.f / sqrtf(ss / (float)D + a.eps);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = x[r] * inv * (is_q ? gq[r] : gk[r]);
      }
      f32x4_t o;
      if (a.layout == 0) {
        o = f32x4_t{x[1], x[0], x[3], x[2]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = __shfl(x[r], other, 64);
      }
      if (turned) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = x[r] * cs[r] + o[r] * sn[r];
      }
      if (h >= nh) continue;
      if (is_q) *reinterpret_cast<f32x4_t*>(row + column(h) + d0) = x;
      else store(kdst + (in_span * a.G + (size_t)(h - a.H)) * D + d0, x, kwide);
    }
  }
  const int nv = a.GV * a.DV;
  for (int e = (blockIdx.y * 256 + threadIdx.x) * 4; e < nv; e += 1024 * gridDim.y) {
    f32x4_t x = *reinterpret_cast<const f32x4_t*>(row + a.v_off + e);
    if (a.vfirst_in) x = (1.f - a.lam) * x + a.lam * *reinterpret_cast<const f32x4_t*>(a.vfirst_in + (size_t)t * a.ldvf + e);
    if (a.vfirst_out) *reinterpret_cast<f32x4_t*>(a.vfirst_out + (size_t)t * a.ldvf + e) = x;
    store(vdst + in_span * nv + e, x, vwide);
  }
}

// ------------------------------------------------------------------------------------------------ convolution + prep + append
// u[c] = sum_j w[j, c] x[t - (taps - 1) + j, c] for the channels [q | k | v] of the rows x (inputs of earlier steps: the slot's tail), then
// the query row and the key row as a whole are divided by their root mean square and weighted, their heads rotated; queries go to q_out,
// keys and values to their pages.  A workgroup per (row, q / k / v); the convolved row is kept in LDS.
struct ConvPrepArgs {
  const float* x; long ld;                     // [T][HD + GD + GV]
  const void* w; const void* qnorm; const void* knorm; int wdt; int taps;      // w: [taps][HD + GD + GV]
  float* tail; int write_tail;                 // [slots][taps - 1][C]; write_tail: every portion has ONE row, which also moves its tail on
  float eps; const float* freq; int rot_dims, pairs; float mag;
  float* q_out; long ldq;
  void* const* kspans; void* const* vspans; int span_stride, span_len, cdt;
  const int32_t* tok_slot; const int32_t* tok_pos; const int32_t* tok_off;
  int HD, GD, GV, D;
};

template <int NT>
__global__ __launch_bounds__(NT) void qkv_conv_prep_append_kernel(ConvPrepArgs a) {
  extern __shared__ float us[];
  __shared__ float cs[128], sn[128], red[NT / 64];
  const int t = blockIdx.x, part = blockIdx.y, tid = threadIdx.x;      // part 0: q, 1: k, 2: v
  const int pos = a.tok_pos[t], off = a.tok_off[t], nt = a.taps - 1, C = a.HD + a.GD + a.GV, half = a.rot_dims >> 1;
  const int c0 = part == 0 ? 0 : (part == 1 ? a.HD : a.HD + a.GD), n = part == 0 ? a.HD : (part == 1 ? a.GD : a.GV);
  const size_t sp = (size_t)a.tok_slot[t] * a.span_stride + pos / a.span_len, in_span = (size_t)(pos % a.span_len);
  float* tl = a.tail ? a.tail + (size_t)a.tok_slot[t] * nt * C : nullptr;
  if (part < 2)
    for (int i = tid; i < half; i += NT) {
      float s, c;
      rope_sincos((uint32_t)pos, a.freq[i], &s, &c);
      sn[i] = s * a.mag;
      cs[i] = c * a.mag;
    }
  float ss = 0.f;
  for (int i = tid; i < n; i += NT) {
    const int c = c0 + i;
    float acc = 0.f;
    for (int k = 0; k < a.taps; ++k) {
      const int d = nt - k, o = off - d;
      const float v = o >= 0 ? a.x[(size_t)(t - d) * a.ld + c] : tl[(size_t)(nt + o) * C + c];
      acc = __builtin_fmaf(ld_any(a.w, (size_t)k * C + c, a.wdt), v, acc);
      if (a.write_tail && k > 0) tl[(size_t)(k - 1) * C + c] = v;      // (off == 0: row k - 1 was read in the turn before)
    }
    ss = __builtin_fmaf(acc, acc, ss);
    if (part < 2) us[i] = acc;
    else st_any(a.vspans[sp], in_span * n + i, a.cdt, acc);
  }
  if (part == 2) return;
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) ss += red[w];
  const float inv = 1.f / sqrtf(ss / (float)n + a.eps);
  const void* gamma = part == 0 ? a.qnorm : a.knorm;
  void* kdst = part == 1 ? a.kspans[sp] : nullptr;
  auto normed = [&](int i) { return gamma ? us[i] * inv * ld_any(gamma, i, a.wdt) : us[i]; };
  for (int i = tid; i < n; i += NT) {
    const int d = i % a.D;
    float y = normed(i);
    if (d < a.rot_dims) {
      const int p = a.pairs ? d >> 1 : (d < half ? d : d - half);
      const bool first = a.pairs ? (d & 1) == 0 : d < half;
      const float o = normed(a.pairs ? (first ? i + 1 : i - 1) : (first ? i + half : i - half));
      y = first ? y * cs[p] - o * sn[p] : y * cs[p] + o * sn[p];
    }
    if (part == 0) a.q_out[(size_t)t * a.ldq + i] = y;
    else st_any(kdst, in_span * n + i, a.cdt, y);
  }
}

// The same for rows of whole 16-byte units (head sizes that are multiples of 4): a thread owns EPT units of 4 channels, all of its loads are
// issued before the first use, the convolved row stays in registers; neighbouring dimensions rotate inside a unit, halves through LDS.
// The number of threads follows the row's length alone: a row's bits do not depend on the batch.
template <int WT>
__device__ __forceinline__ f32x4_t load_w4(const void* p, size_t i) {
  if constexpr (WT == DIHIP_F32) return *reinterpret_cast<const f32x4_t*>((const float*)p + i);
  const u32x2_t r = *reinterpret_cast<const u32x2_t*>((const uint16_t*)p + i);
  return f32x4_t{__uint_as_float(r[0] << 16), __uint_as_float(r[0] & 0xffff0000u), __uint_as_float(r[1] << 16), __uint_as_float(r[1] & 0xffff0000u)};
}
__device__ __forceinline__ void store4(void* p, size_t i, int dt, const f32x4_t& v) {
  if (dt == DIHIP_F32) *reinterpret_cast<f32x4_t*>((float*)p + i) = v;
  else *reinterpret_cast<u32x2_t*>((uint16_t*)p + i) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

template <int WT, int NT, int EPT>
__global__ __launch_bounds__(NT) void qkv_conv_prep_append_vec_kernel(ConvPrepArgs a) {
  extern __shared__ float us[];                                         // halves: the normed row
  __shared__ float cs[128], sn[128], red[NT / 64];
  const int t = blockIdx.x, part = blockIdx.y, tid = threadIdx.x;      // part 0: q, 1: k, 2: v
  const int nt = a.taps - 1, C = a.HD + a.GD + a.GV, half = a.rot_dims >> 1;
  const int c0 = part == 0 ? 0 : (part == 1 ? a.HD : a.HD + a.GD), n = part == 0 ? a.HD : (part == 1 ? a.GD : a.GV);
  if (tid * 4 >= n && tid >= 64 * ((n / 4 + 63) / 64) && part == 2) return;      // (values: no barrier follows; whole waves past the row)
  const int pos = a.tok_pos[t], off = a.tok_off[t], slot = a.tok_slot[t];
  float* tl = a.tail ? a.tail + (size_t)slot * nt * C : nullptr;
  int c[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) c[e] = min((tid + e * NT) * 4, n - 4);          // units past the row repeat its last one and are not stored
  f32x4_t u[EPT], gm[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) u[e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const void* gamma = part == 0 ? a.qnorm : (part == 1 ? a.knorm : nullptr);
  if (gamma) {
#pragma unroll
    for (int e = 0; e < EPT; ++e) gm[e] = load_w4<WT>(gamma, c[e]);
  }
  for (int k0 = 0; k0 < a.taps; k0 += 4) {
    f32x4_t xv[4][EPT], wv[4][EPT];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int k = min(k0 + kk, a.taps - 1), d = nt - k, o = off - d;
      const float* src = o >= 0 ? a.x + (size_t)(t - d) * a.ld + c0 : tl + (size_t)(nt + o) * C + c0;
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        xv[kk][e] = *reinterpret_cast<const f32x4_t*>(src + c[e]);
        wv[kk][e] = load_w4<WT>(a.w, (size_t)k * C + c0 + c[e]);
      }
    }
    if (k0 == 0 && part < 2 && tid < half) {       // while the loads are in flight
      float s_, c_;
      rope_sincos((uint32_t)pos, a.freq[tid], &s_, &c_);
      sn[tid] = s_ * a.mag;
      cs[tid] = c_ * a.mag;
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (k0 + kk < a.taps) {
#pragma unroll
        for (int e = 0; e < EPT; ++e) {
#pragma unroll
          for (int x = 0; x < 4; ++x) u[e][x] = __builtin_fmaf(wv[kk][e][x], xv[kk][e][x], u[e][x]);
          if (a.write_tail && k0 + kk > 0 && (tid + e * NT) * 4 < n)      // tail row k - 1 <- the input of tap k (row k - 1 has been read)
            *reinterpret_cast<f32x4_t*>(tl + (size_t)(k0 + kk - 1) * C + c0 + c[e]) = xv[kk][e];
        }
      }
    }
  }
  const size_t sp = (size_t)slot * a.span_stride + pos / a.span_len, in_span = (size_t)(pos % a.span_len);
  if (part == 2) {
    void* vdst = a.vspans[sp];
#pragma unroll
    for (int e = 0; e < EPT; ++e)
      if ((tid + e * NT) * 4 < n) store4(vdst, in_span * n + c[e], a.cdt, u[e]);
    return;
  }
  void* kdst = part == 1 ? a.kspans[sp] : nullptr;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < EPT; ++e)
    if ((tid + e * NT) * 4 < n) {
#pragma unroll
      for (int x = 0; x < 4; ++x) ss = __builtin_fmaf(u[e][x], u[e][x], ss);
    }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  if (gamma) {
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) ss += red[w];
    const float inv = 1.f / sqrtf(ss / (float)n + a.eps);
#pragma unroll
    for (int e = 0; e < EPT; ++e)
#pragma unroll
      for (int x = 0; x < 4; ++x) u[e][x] = u[e][x] * inv * gm[e][x];
  }
  if (half && !a.pairs) {
#pragma unroll
    for (int e = 0; e < EPT; ++e)
      if ((tid + e * NT) * 4 < n) *reinterpret_cast<f32x4_t*>(&us[c[e]]) = u[e];
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    if ((tid + e * NT) * 4 >= n) continue;
    const int d0 = c[e] % a.D;
    f32x4_t y = u[e];
    if (d0 < a.rot_dims) {
      if (a.pairs) {
#pragma unroll
        for (int x = 0; x < 4; x += 2)
          if (d0 + x < a.rot_dims) {
            const int p = (d0 + x) >> 1;
            y[x] = u[e][x] * cs[p] - u[e][x + 1] * sn[p];
            y[x + 1] = u[e][x + 1] * cs[p] + u[e][x] * sn[p];
          }
      } else {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int d = d0 + x;
          if (d < half) y[x] = u[e][x] * cs[d] - us[c[e] + x + half] * sn[d];
          else if (d < a.rot_dims) y[x] = u[e][x] * cs[d - half] + us[c[e] + x - half] * sn[d - half];
        }
      }
    }
    if (part == 0) *reinterpret_cast<f32x4_t*>(a.q_out + (size_t)t * a.ldq + c[e]) = y;
    else store4(kdst, in_span * n + c[e], a.cdt, y);
  }
}

// ------------------------------------------------------------------------------------------------ f32 row kernel
struct GqaArgs {
  void* out; int odt; long ldo;
  const float* q; long ldq;
  void* const* kspans; void* const* vspans; int span_stride, span_len;
  const void* sink; int wdt, sink_mode;   // 0: none, 1: sink[h], 2: the constant 0
  float softcap;                          // <= 0: none
  const float* gate; long ldg;            // [T, H] multiplier (NULL: none; ldg 0: one row for all)
  const int32_t* tok_slot; const int32_t* tok_pos; const int32_t* ent_slot; const int32_t* ent_row0; const int32_t* ent_count;
  int H, G, D, DV; float scale;
  float* ws; int rows_total;
  int maps, window, keep_first;           // window <= 0: every key up to the row's own
};

__device__ __forceinline__ float cap_score(float s, float cap) { return cap > 0.f ? cap * tanhf(s / cap) : s; }

// One workgroup per row, its 4 waves take the (head, map) pairs in turn; a wave walks the keys it may read 64 at a time (first the
// kept first keys that lie before the window, then the window): lane j scores key j (d ascending), the chunk joins the running
// softmax, then the lanes turn to the value elements and add the weighted rows.
template <int CT, int RV>
__global__ __launch_bounds__(256) void gqa_attn_kernel(GqaArgs a) {
  __shared__ float qs[4][256];
  __shared__ float ps[4][64];
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pos = a.tok_pos[t], H = a.H, G = a.G, D = a.D, DV = a.DV, hpg = H / G, M = a.maps, HQ = H * M, GK = G * M;
  const int w_lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;   // the window is [w_lo, pos]
  const int first_hi = min(a.keep_first, w_lo);                     // the kept first keys before it: [0, first_hi)
  void* const* ktab = a.kspans + (size_t)a.tok_slot[t] * a.span_stride;
  void* const* vtab = a.vspans + (size_t)a.tok_slot[t] * a.span_stride;
  constexpr size_t ES = CT == DIHIP_F32 ? 4 : 2;
  for (int h0 = 0; h0 < HQ; h0 += 4) {
    const int hq = h0 + wave;
    const bool live = hq < HQ;
    const int h = (live ? hq : 0) / M, mp = (live ? hq : 0) - h * M;
    const int g = h / hpg, gk = g * M + mp;
    __syncthreads();
    if (live)
      for (int d = lane; d < D; d += 64) qs[wave][d] = a.q[(size_t)t * a.ldq + (size_t)hq * D + d];
    __syncthreads();
    float mx = -INFINITY, den = 0.f;
    if (a.sink_mode == 1) { mx = ld_any(a.sink, h, a.wdt); den = 1.f; }
    else if (a.sink_mode == 2) { mx = 0.f; den = 1.f; }
    float acc[RV];
#pragma unroll
    for (int v = 0; v < RV; ++v) acc[v] = 0.f;
    for (int part = 0; part < 2; ++part) {                       // the same trip counts in every wave of the block
      const int r_lo = part ? w_lo : 0, r_hi = part ? pos + 1 : first_hi;
      for (int j0 = r_lo; j0 < r_hi; j0 += 64) {
        const int j = j0 + lane;
        const bool valid = live && j < r_hi;
        float s = -INFINITY;
        if (valid) {
          const char* kr = (const char*)ktab[j / a.span_len] + ((size_t)(j % a.span_len) * GK + gk) * D * ES;
          float d = 0.f;
          for (int r = 0; r < D; ++r) d = __builtin_fmaf(qs[wave][r], load_ft<CT>(kr, r), d);
          s = cap_score(d * a.scale, a.softcap);
        }
        const float mnew = fmaxf(mx, wave_max(s));
        const float corr = mx == -INFINITY ? 0.f : expf(mx - mnew);
        const float p = valid ? expf(s - mnew) : 0.f;
        den = den * corr + wave_sum(p);
#pragma unroll
        for (int v = 0; v < RV; ++v) acc[v] *= corr;
        mx = mnew;
        ps[wave][lane] = p;
        __syncthreads();
        if (live) {
          const int cnt = min(64, r_hi - j0);
          for (int jj = 0; jj < cnt; ++jj) {
            const int jk = j0 + jj;
            const char* vr = (const char*)vtab[jk / a.span_len] + ((size_t)(jk % a.span_len) * G + g) * DV * ES;
            const float pj = ps[wave][jj];
#pragma unroll
            for (int v = 0; v < RV; ++v) {
              const int r = v * 64 + lane;
              if (r < DV) acc[v] = __builtin_fmaf(pj, load_ft<CT>(vr, r), acc[v]);
            }
          }
        }
        __syncthreads();
      }
    }
    if (live) {
      const float gt = a.gate ? a.gate[(size_t)t * a.ldg + h] : 1.f;
#pragma unroll
      for (int v = 0; v < RV; ++v) {
        const int r = v * 64 + lane;
        if (r < DV) st_any(a.out, (size_t)t * a.ldo + (size_t)hq * DV + r, a.odt, acc[v] / den * gt);
      }
    }
  }
}

// Two maps per head -> one: d = first - lam * second, out = d / sqrt(mean(d^2) + eps) * out_scale.  A wave per (row, head).
__global__ __launch_bounds__(256) void maps_diff_norm_kernel(void* __restrict__ y, int ydt, long ldy, const float* __restrict__ x, long ldx,
                                                             float lam, float out_scale, float eps, int TH, int H, int DV) {
  const int pair = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (pair >= TH) return;
  const int t = pair / H, h = pair - t * H;
  const float* a1 = x + (size_t)t * ldx + (size_t)h * 2 * DV;
  const float* a2 = a1 + DV;
  float v[8], ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int d = lane + 64 * i;
    v[i] = d < DV ? a1[d] - lam * a2[d] : 0.f;
    ss = __builtin_fmaf(v[i], v[i], ss);
  }
  const float inv = out_scale / sqrtf(wave_sum(ss) / (float)DV + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int d = lane + 64 * i;
    if (d < DV) st_any(y, (size_t)t * ldy + (size_t)h * DV + d, ydt, v[i] * inv);
  }
}

// ------------------------------------------------------------------------------------------------ matrix-core kernel
// A workgroup owns 64 consecutive (row, query head) pairs of ONE portion, ONE key/value head and ONE map -- 16 per wave -- and
// walks the 32-key tiles those pairs can see (with a window: the tiles of the kept first keys, then those from the window of its
// first row on).  Per tile: S^T = K . Q^T (the tile's key rows as they lie in LDS against the wave's
// query fragments, held in registers for the whole walk), cap + mask + running softmax on the accumulator lanes, then
// O^T += V^T . P^T with P straight from those lanes and V^T read from the value tile through the transposing LDS read.  The
// next tile's rows are in flight meanwhile.  Head sizes that are no multiple of the tile's granule are padded with zero
// columns in LDS.  The key walk can be split over gridDim.z workgroups; the partial records are merged by a second launch.
__device__ __forceinline__ f32x4_t mfma_bf16g(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ float fast_tanh(float x) { return 1.f - 2.f / (1.f + __expf(2.f * x)); }

template <int DMAX, int VMAX>
__global__ __launch_bounds__(256) void gqa_attn_mc_kernel(GqaArgs a) {
  constexpr int KS = DMAX / 32, DT = VMAX / 16, UNK = DMAX / 64, UNV = VMAX / 64;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int G = a.G, H = a.H, D = a.D, DV = a.DV, hpg = H / G;
  const int M = a.maps, GK = G * M;
  const int e = blockIdx.y / GK, gk = blockIdx.y - e * GK, g = gk / M, mp = gk - g * M, split = blockIdx.z, nsplit = gridDim.z;
  const int cnt = a.ent_count[e], row0 = a.ent_row0[e];
  const int nrows = cnt * hpg, r0 = blockIdx.x * 64;
  if (r0 >= nrows) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ni = lane & 15, kb = lane >> 4;
  const int Dp = (D + 31) & ~31, Vp = (DV + 15) & ~15;
  const int pitchk = (Dp + 8) * 2, pitchv = (Vp + 8) * 2;
  unsigned char* ksm = smem;
  unsigned char* vsm = smem + 32 * pitchk;
  const int pos0 = a.tok_pos[row0];
  const int myrow = r0 + wave * 16 + ni;
  const bool row_ok = myrow < nrows;
  const int rr = row_ok ? myrow : nrows - 1;
  const int tq = rr / hpg, h = g * hpg + (rr - tq * hpg), hq = h * M + mp, p = pos0 + tq;
  const int p_lo = pos0 + r0 / hpg, p_hi = pos0 + min(r0 + 63, nrows - 1) / hpg;
  const int tile_hi = p_hi >> 5;
  const int win_t0 = (a.window > 0 ? max(0, p_lo - a.window + 1) : 0) >> 5;          // the first tile of the window of the first row
  const int n_first = min(win_t0, (min(a.keep_first, p_hi + 1) + 31) >> 5);           // tiles of kept first keys before it
  const int n_tiles = n_first + tile_hi - win_t0 + 1;
  const int per = (n_tiles + nsplit - 1) / nsplit;
  const int my_lo = split * per, my_hi = min(n_tiles - 1, my_lo + per - 1);           // indices into the walk: tile_of(i)
  auto tile_of = [&](int i) { return i < n_first ? i : win_t0 + (i - n_first); };

  u32x4_t qf[KS];
  {
    const float* qrow = a.q + (size_t)(row0 + tq) * a.ldq + (size_t)hq * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = u32x4_t{0u, 0u, 0u, 0u};
      const int d0 = ks * 32 + kb * 8;
      if (d0 < D) {   // D % 8 == 0: a unit of 8 is inside or outside
        const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(qrow + d0);
        const f32x4_t hi = *reinterpret_cast<const f32x4_t*>(qrow + d0 + 4);
        qf[ks] = u32x4_t{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]), pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
      }
    }
  }
  const bool with_sink = a.sink_mode != 0 && split == 0;
  float m = with_sink ? (a.sink_mode == 1 ? ld_any(a.sink, h, a.wdt) : 0.f) : -1e30f;
  float l = with_sink ? 1.f : 0.f;
  const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) oacc[t] = z4;

  // zero the padding columns once: the tiles' stores never touch them
  for (int i = tid; i < 32 * (Dp - D + 8); i += 256) {
    const int kin = i / (Dp - D + 8), c = D + i % (Dp - D + 8);
    reinterpret_cast<uint16_t*>(ksm + kin * pitchk)[c] = 0;
  }
  for (int i = tid; i < 32 * (Vp - DV + 8); i += 256) {
    const int kin = i / (Vp - DV + 8), c = DV + i % (Vp - DV + 8);
    reinterpret_cast<uint16_t*>(vsm + kin * pitchv)[c] = 0;
  }
  __shared__ const char* ktabs[128];
  __shared__ const char* vtabs[128];
  void* const* gkp = a.kspans + (size_t)a.ent_slot[e] * a.span_stride;
  void* const* gv = a.vspans + (size_t)a.ent_slot[e] * a.span_stride;
  const int span_lo = my_lo <= my_hi ? (tile_of(my_lo) * 32) / a.span_len : 0;
  for (int i = tid; i < 128; i += 256) {
    const int sp = span_lo + i;
    const bool in = sp * a.span_len <= p_hi;
    ktabs[i] = in ? (const char*)gkp[sp] : nullptr;
    vtabs[i] = in ? (const char*)gv[sp] : nullptr;
  }
  __syncthreads();
  const int uprk = D >> 3, uprv = DV >> 3;
  int gok[UNK], lok[UNK], gov[UNV], lov[UNV];
#pragma unroll
  for (int j = 0; j < UNK; ++j) {
    const int u = tid + 256 * j, kin = u / uprk, c8 = u - kin * uprk;
    gok[j] = kin < 32 ? ((kin * GK + gk) * D + c8 * 8) * 2 : -1;
    lok[j] = kin * pitchk + c8 * 16;
  }
#pragma unroll
  for (int j = 0; j < UNV; ++j) {
    const int u = tid + 256 * j, kin = u / uprv, c8 = u - kin * uprv;
    gov[j] = kin < 32 ? ((kin * G + g) * DV + c8 * 8) * 2 : -1;
    lov[j] = kin * pitchv + c8 * 16;
  }
  u32x4_t prek[UNK], prev[UNV];
  auto fetch = [&](int tile) {
    const int key0 = tile * 32, sp = key0 / a.span_len, in = key0 - sp * a.span_len;
    const bool near = sp - span_lo < 128;
    const char* kbp = (near ? ktabs[sp - span_lo] : (const char*)gkp[sp]) + (size_t)in * GK * D * 2;
    const char* vbp = (near ? vtabs[sp - span_lo] : (const char*)gv[sp]) + (size_t)in * G * DV * 2;
#pragma unroll
    for (int j = 0; j < UNK; ++j) {
      prek[j] = u32x4_t{0u, 0u, 0u, 0u};
      if (gok[j] >= 0) prek[j] = gload<u32x4_t>(kbp + gok[j]);
    }
#pragma unroll
    for (int j = 0; j < UNV; ++j) {
      prev[j] = u32x4_t{0u, 0u, 0u, 0u};
      if (gov[j] >= 0) prev[j] = gload<u32x4_t>(vbp + gov[j]);
    }
  };
  if (my_lo <= my_hi) fetch(tile_of(my_lo));
  for (int ti = my_lo; ti <= my_hi; ++ti) {
    const int tile = tile_of(ti);
#pragma unroll
    for (int j = 0; j < UNK; ++j)
      if (gok[j] >= 0) *reinterpret_cast<u32x4_t*>(ksm + lok[j]) = prek[j];
#pragma unroll
    for (int j = 0; j < UNV; ++j)
      if (gov[j] >= 0) *reinterpret_cast<u32x4_t*>(vsm + lov[j]) = prev[j];
    __syncthreads();
    if (ti + 1 <= my_hi) fetch(tile_of(ti + 1));
    f32x4_t sacc[2] = {z4, z4};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks * 32 < D) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(ksm + (nt * 16 + ni) * pitchk + (ks * 32 + kb * 8) * 2);
          sacc[nt] = mfma_bf16g(kf, qf[ks], sacc[nt]);
        }
      }
    }
    float sv[2][4], mx = -INFINITY;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = tile * 32 + nt * 16 + kb * 4 + r;
        float s = sacc[nt][r] * a.scale;
        if (a.softcap > 0.f) s = a.softcap * fast_tanh(s / a.softcap);
        const bool seen = key <= p && (a.window <= 0 || p - key < a.window || key < a.keep_first);
        sv[nt][r] = seen ? s : -INFINITY;
        mx = fmaxf(mx, sv[nt][r]);
      }
    mx = rows_max(mx);
    const float mn = fmaxf(m, mx);
    const float corr = __expf(m - mn);
    m = mn;
    float psum = 0.f, ev[2][4];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ev[nt][r] = __expf(sv[nt][r] - mn);
        psum += ev[nt][r];
      }
    l = l * corr + rows_sum(psum);
    const u32x4_t pf = {pack_bf16x2(ev[0][0], ev[0][1]), pack_bf16x2(ev[0][2], ev[0][3]), pack_bf16x2(ev[1][0], ev[1][1]),
                        pack_bf16x2(ev[1][2], ev[1][3])};
    if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0ull) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) oacc[t][r] *= corr;
    }
    const unsigned char* tr0 = vsm + (kb * 4 + (ni >> 2)) * pitchv + (ni & 3) * 8;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      if (t * 16 < DV) {
        const u32x2_t lo2 = lds_read_tr16(tr0 + t * 32);
        const u32x2_t hi2 = lds_read_tr16(tr0 + t * 32 + 16 * pitchv);
        const u32x4_t vf = {lo2[0], lo2[1], hi2[0], hi2[1]};
        oacc[t] = mfma_bf16g(vf, pf, oacc[t]);
      }
    }
    __syncthreads();
  }
  asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
  if (!row_ok) return;
  if (nsplit == 1) {
    const float inv = (a.gate ? a.gate[(size_t)(row0 + tq) * a.ldg + h] : 1.f) / l;
    const size_t o = (size_t)(row0 + tq) * a.ldo + (size_t)hq * DV + kb * 4;
#pragma unroll
    for (int t = 0; t < DT; ++t)
      if (t * 16 + kb * 4 < DV) store4(a.out, o + t * 16, a.odt, f32x4_t{oacc[t][0] * inv, oacc[t][1] * inv, oacc[t][2] * inv, oacc[t][3] * inv});
  } else {
    float* o = a.ws + ((size_t)split * a.rows_total + (size_t)(row0 + tq) * H * M + hq) * (Vp + 4);
#pragma unroll
    for (int t = 0; t < DT; ++t)
      if (t * 16 < Vp) *reinterpret_cast<f32x4_t*>(o + t * 16 + kb * 4) = oacc[t];
    if (kb == 0) { o[Vp] = m; o[Vp + 1] = l; }
  }
}

// The same for head sizes of exactly 64 or 128 and pages of whole 64-key tiles (D / DV compile-time: no guard inside the walk).
//   * a workgroup owns 64 * MT (row, query head) pairs, 16 * MT per wave: with MT = 2 every key and value operand read from LDS serves two products;
//   * 64-key tiles go straight into LDS (global_load_lds, two copies): the loads of the next tile are issued behind the one barrier of a tile and
//     have that tile's time to land.  The 16-byte chunks of a row change places on the memory side (keys: chunk ^ key; values: pairs
//     of chunks ^ key), so that neither the operand reads nor the transposing reads meet in a bank;
//   * the mask is looked at only in tiles where some pair of the wave does not see every key; exp2 with the scale folded in;
//   * row tiles are dealt so that the two workgroups a CU holds have together the same walk (up to 512 of them), else longest first.
// A portion of 2048 rows, 32 heads of 128 over 8 key heads: 300 -> 77 us (115 -> 447 TFLOP/s; with capped scores 89); 500 rows beside 13 decoded ones, 16
// heads over 4: 139 -> 21; 24 decoded rows at 160 .. 700 keys, five splits: 21 -> 11.  The kernel above, which tests the head sizes inside the walk,
// waited for every tile's loads.  What bounds this one is the instruction stream between the products (softmax: ~180 vector
// instructions per 64 products).
template <int D, int DV, int MT, bool CAP>
__global__ __launch_bounds__(256, 2) void gqa_attn_tile_kernel(GqaArgs a, int gx) {
  constexpr int KS = D / 32, DT = DV / 16, NT = 4, TABLE = 128;
  constexpr int KROW = D * 2, VROW = DV * 2, KBYTES = 64 * KROW, VBYTES = 64 * VROW, COPY = KBYTES + VBYTES;
  constexpr int KPP = 1024 / KROW, VPP = 1024 / VROW;                 // keys per 1 KiB piece
  constexpr int KPW = 64 / KPP / 4, VPW = 64 / VPP / 4;               // pieces per wave and tile: piece wave + 4 j
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ const char* ktabs[TABLE];
  __shared__ const char* vtabs[TABLE];
  const int G = a.G, H = a.H, hpg = H / G, M = a.maps, GK = G * M, gy = gridDim.x / gx;
  // linear index -> (row tile, portion and key head)
  int tile_x, ey;
  {
    const int lin = blockIdx.x, total = gridDim.x;
    const int order = total <= 512 && lin >= total / 2 ? lin - total / 2 : total - 1 - lin;
    tile_x = order / gy;
    ey = order - tile_x * gy;
  }
  const int e = ey / GK, gk = ey - e * GK, g = gk / M, mp = gk - g * M, split = blockIdx.z, nsplit = gridDim.z;
  const int cnt = a.ent_count[e], row0 = a.ent_row0[e];
  const int nrows = cnt * hpg, r0 = tile_x * (64 * MT);
  if (r0 >= nrows) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ni = lane & 15, kb = lane >> 4;
  const int pos0 = a.tok_pos[row0], end = pos0 + cnt - 1;             // the sequence's last position
  const int p_lo = pos0 + r0 / hpg, p_hi = pos0 + min(r0 + 64 * MT - 1, nrows - 1) / hpg;
  const int win_t0 = (a.window > 0 ? max(0, p_lo - a.window + 1) : 0) >> 6;
  const int n_first = min(win_t0, (min(a.keep_first, p_hi + 1) + 63) >> 6);
  const int n_tiles = n_first + (p_hi >> 6) - win_t0 + 1;
  const int per = (n_tiles + nsplit - 1) / nsplit;
  const int my_lo = split * per, my_hi = min(n_tiles - 1, my_lo + per - 1);
  auto tile_of = [&](int i) { return i < n_first ? i : win_t0 + (i - n_first); };
  // this wave's pairs
  const int w0 = r0 + wave * 16 * MT;
  const int wp_lo = pos0 + min(w0, nrows - 1) / hpg, wp_hi = pos0 + min(w0 + 16 * MT - 1, nrows - 1) / hpg;   // positions of its first and last pair
  const bool wave_on = w0 < nrows;
  int hq[MT], tq[MT], h[MT];
  bool ok[MT];
  u32x4_t qf[MT][KS];
  f32x4_t oacc[MT][DT];
  float m[MT], l[MT];
  constexpr float LOG2E = 1.44269504088896341f;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r = w0 + i * 16 + ni, rr = min(r, nrows - 1);
    ok[i] = r < nrows;
    tq[i] = rr / hpg;
    h[i] = g * hpg + (rr - tq[i] * hpg);
    hq[i] = h[i] * M + mp;
    const float* qrow = a.q + (size_t)(row0 + tq[i]) * a.ldq + (size_t)hq[i] * D + kb * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(qrow + ks * 32), hi = *reinterpret_cast<const f32x4_t*>(qrow + ks * 32 + 4);
      qf[i][ks] = u32x4_t{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]), pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
    }
    const bool with_sink = a.sink_mode != 0 && split == 0;
    m[i] = with_sink ? (a.sink_mode == 1 ? ld_any(a.sink, h[i], a.wdt) * LOG2E : 0.f) : -1e30f;      // scores and maxima: times log2 e
    l[i] = with_sink && kb == 0 ? 1.f : 0.f;                            // (a lane's own keys: summed over kb at the end)
#pragma unroll
    for (int t = 0; t < DT; ++t) oacc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  void* const* gkp = a.kspans + (size_t)a.ent_slot[e] * a.span_stride;
  void* const* gv = a.vspans + (size_t)a.ent_slot[e] * a.span_stride;
  // span pointers of the walk, TABLE at a time
  auto fill = [&](int first) {
    for (int i = tid; i < TABLE; i += 256) {
      const bool in = (long)(first + i) * a.span_len <= p_hi;
      ktabs[i] = in ? (const char*)gload<void*>(gkp + first + i) : nullptr;
      vtabs[i] = in ? (const char*)gload<void*>(gv + first + i) : nullptr;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
  };
  int table0 = my_lo <= my_hi ? tile_of(my_lo) * 64 / a.span_len : 0;
  fill(table0);
  // where this lane's 16 bytes of a piece come from
  const int kk = lane / (KROW / 16), kc = lane % (KROW / 16), vk = lane / (VROW / 16), vc = lane % (VROW / 16);
  const int kkey = wave * KPP + kk, vkey = wave * VPP + vk;            // key of piece `wave`; piece wave + 4 j: 4 j KPP further
  const uint32_t koff = (uint32_t)(kkey * GK + gk) * KROW + (uint32_t)((kc ^ (D == 128 ? kkey & 15 : kkey & 7)) * 16);
  const uint32_t voff = (uint32_t)(vkey * G + g) * VROW + (uint32_t)((vc ^ (DV == 128 ? (vkey & 7) * 2 : ((vkey >> 1) & 3) * 2)) * 16);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * 1024;
  auto fetch = [&](int i, int copy) {
    const int key0 = tile_of(i) * 64, sp = key0 / a.span_len, in = key0 - sp * a.span_len;
    if (sp - table0 >= TABLE || sp < table0) {    // (uniform)
      __syncthreads();
      table0 = sp;
      fill(table0);
    }
    const uint64_t ka = (uint64_t)ktabs[sp - table0], va = (uint64_t)vtabs[sp - table0];
    const uint64_t ku = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)ka) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(ka >> 32)) << 32;
    const uint64_t vu = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)va) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(va >> 32)) << 32;
    const char* kp = (const char*)ku + (size_t)in * GK * KROW;
    const char* vp = (const char*)vu + (size_t)in * G * VROW;
#pragma unroll
    for (int j = 0; j < KPW; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + copy * COPY + j * 4096), "v"(koff),
                   "s"(kp + (size_t)j * 4 * KPP * GK * KROW) : "memory");
#pragma unroll
    for (int j = 0; j < VPW; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + copy * COPY + KBYTES + j * 4096), "v"(voff),
                   "s"(vp + (size_t)j * 4 * VPP * G * VROW) : "memory");
  };
  // operand addresses: keys nt * 16 + ni, chunks ks * 4 + kb; values rows kb * 4 + ni / 4 (+ 16, + 32 ..), chunks 2 t + ni % 4 / 2
  int kfo[KS], vfo[DT];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kfo[ks] = ni * KROW + (((ks * 4 + kb) ^ (D == 128 ? ni : ni & 7)) * 16);
  {
    const int vr = kb * 4 + (ni >> 2), f = DV == 128 ? (vr & 7) * 2 : ((vr >> 1) & 3) * 2;
#pragma unroll
    for (int t = 0; t < DT; ++t) vfo[t] = KBYTES + vr * VROW + (((2 * t) ^ f) + ((ni & 3) >> 1)) * 16 + (ni & 1) * 8;
  }
  const float sl2 = a.scale * LOG2E, cap = a.softcap, cap_in = CAP ? 2.f * a.scale * LOG2E / cap : 0.f, cap2 = cap * LOG2E;
  if (my_lo <= my_hi) fetch(my_lo, 0);
  for (int ti = my_lo; ti <= my_hi; ++ti) {
    const int copy = (ti - my_lo) & 1, key0 = tile_of(ti) * 64;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();     // the tile has landed; the other copy has been read
    asm volatile("" ::: "memory");
    if (ti + 1 <= my_hi) fetch(ti + 1, copy ^ 1);
    const unsigned char* base = smem + copy * COPY;
    if (key0 + 63 > end) {            // (uniform) rows that no token has written: an infinity there would reach the sums through a weight of 0
      for (int i = tid; i < (key0 + 63 - end) * (VROW / 16); i += 256)
        *reinterpret_cast<u32x4_t*>(const_cast<unsigned char*>(base) + KBYTES + (size_t)(end + 1 - key0) * VROW + i * 16) = u32x4_t{0u, 0u, 0u, 0u};
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (!wave_on || key0 > wp_hi) continue;
    if (a.window > 0 && key0 + 63 <= wp_lo - a.window && key0 >= a.keep_first) continue;   // before every window of the wave
    f32x4_t sacc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) sacc[i][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4_t kf[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) kf[nt] = *reinterpret_cast<const u32x4_t*>(base + kfo[ks] + nt * 16 * KROW);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < MT; ++i) sacc[i][nt] = mfma_bf16g(kf[nt], qf[i][ks], sacc[i][nt]);
    }
    const bool whole = key0 + 63 <= wp_lo && (a.window <= 0 || wp_hi - key0 < a.window || key0 + 63 < a.keep_first);   // (uniform)
    u32x4_t pf[MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int p = pos0 + tq[i];
      float mx = -INFINITY;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float s;
          if constexpr (CAP) s = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(sacc[i][nt][r] * cap_in));   // cap * tanh(s / cap)
          else s = sacc[i][nt][r] * sl2;
          if (!whole) {
            const int key = key0 + nt * 16 + kb * 4 + r;
            if (!(key <= p && (a.window <= 0 || p - key < a.window || key < a.keep_first))) s = -INFINITY;
          }
          sacc[i][nt][r] = s;
          mx = fmaxf(mx, s);
        }
      mx = fmaxf(m[i], rows_max(mx));
      const float corr = __builtin_amdgcn_exp2f(m[i] - mx);
      m[i] = mx;
      float ps = 0.f;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sacc[i][nt][r] = __builtin_amdgcn_exp2f(sacc[i][nt][r] - mx);
          ps += sacc[i][nt][r];
        }
      l[i] = l[i] * corr + ps;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
        pf[i][hh] = u32x4_t{pack_bf16x2(sacc[i][2 * hh][0], sacc[i][2 * hh][1]), pack_bf16x2(sacc[i][2 * hh][2], sacc[i][2 * hh][3]),
                            pack_bf16x2(sacc[i][2 * hh + 1][0], sacc[i][2 * hh + 1][1]), pack_bf16x2(sacc[i][2 * hh + 1][2], sacc[i][2 * hh + 1][3])};
      if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0ull) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) oacc[i][t][r] *= corr;
      }
    }
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const u32x2_t lo2 = lds_read_tr16(base + vfo[t] + hh * 32 * VROW), hi2 = lds_read_tr16(base + vfo[t] + hh * 32 * VROW + 16 * VROW);
        const u32x4_t vf = {lo2[0], lo2[1], hi2[0], hi2[1]};
#pragma unroll
        for (int i = 0; i < MT; ++i) oacc[i][t] = mfma_bf16g(vf, pf[i][hh], oacc[i][t]);
      }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing may be on its way into LDS when the workgroup leaves
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const float den = rows_sum(l[i]);
    if (!ok[i]) continue;
    if (nsplit == 1) {
      const float inv = (a.gate ? a.gate[(size_t)(row0 + tq[i]) * a.ldg + h[i]] : 1.f) / den;
      const size_t o = (size_t)(row0 + tq[i]) * a.ldo + (size_t)hq[i] * DV + kb * 4;
#pragma unroll
      for (int t = 0; t < DT; ++t)
        store4(a.out, o + t * 16, a.odt, f32x4_t{oacc[i][t][0] * inv, oacc[i][t][1] * inv, oacc[i][t][2] * inv, oacc[i][t][3] * inv});
    } else {   // [split][row, query vector][DV sums, maximum, denominator, ..]
      const int gi = (row0 + tq[i]) * H * M + hq[i];
      float* o = a.ws + ((size_t)split * a.rows_total + gi) * (DV + 4);
#pragma unroll
      for (int t = 0; t < DT; ++t) *reinterpret_cast<f32x4_t*>(o + t * 16 + kb * 4) = oacc[i][t];
      if (kb == 0) { o[DV] = m[i] * 0.69314718055994531f; o[DV + 1] = den; }
    }
  }
}

// The splits' (maximum, denominator, sums) records of one (row, query vector) -> column threadIdx.x of its softmax-weighted sum
// (0 for threads past DV; DV <= 256).  wgt / red: LDS scratch of the workgroup; the call synchronises it.
__device__ __forceinline__ float merge_splits(const float* __restrict__ base, size_t stride, int nsplit, int Vp, int DV, float* wgt, float* red) {
  const int r = min((int)threadIdx.x, DV - 1);
  // the sums of eight splits on their way beside the records' maxima (a loop behind those waits a second time, and for each of the splits past a multiple of its step: six splits of 32 heads 1.3 us more)
  float part[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) part[i] = base[min(i, nsplit - 1) * stride + r];
  float mloc[4], lloc[4], mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int s = threadIdx.x + i * 256;
    mloc[i] = s < nsplit ? base[s * stride + Vp] : -INFINITY;
    lloc[i] = s < nsplit ? base[s * stride + Vp + 1] : 0.f;
    mx = fmaxf(mx, mloc[i]);
  }
  mx = wave_max(mx);
  __syncthreads();                   // wgt / red of an earlier call are no longer read
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float den = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int s = threadIdx.x + i * 256;
    const float w = s < nsplit ? expf(mloc[i] - mx) : 0.f;
    if (s < nsplit) wgt[s] = w;
    den = __builtin_fmaf(w, lloc[i], den);
  }
  den = block256_sum(den, red);      // (its barriers publish wgt)
  float acc = 0.f;
  for (int s0 = 0; s0 < nsplit; s0 += 8) {
    float next[8] = {};
    if (s0 + 8 < nsplit)     // (uniform) the next eight while these are added: attention of 4000 keys in 63 splits, heads of 96, 18.4 us without, 16.1
#pragma unroll
      for (int i = 0; i < 8; ++i) next[i] = base[min(s0 + 8 + i, nsplit - 1) * stride + r];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (s0 + i < nsplit) acc = __builtin_fmaf(wgt[s0 + i], part[i], acc);
      part[i] = next[i];
    }
  }
  return threadIdx.x < DV ? acc / den : 0.f;
}

// one workgroup per (row, query vector); row0: the rows' numbers (NULL: 0, 1, ..)
__global__ __launch_bounds__(256) void gqa_attn_merge_kernel(void* __restrict__ out, int odt, long ldo, const float* __restrict__ ws, int nsplit,
                                                             int rows_total, int H, int maps, int DV, int Vp, const float* __restrict__ gate, long ldg,
                                                             const int32_t* __restrict__ row0) {
  __shared__ float wgt[1024];
  __shared__ float red[4];
  const int HQ = H * maps, u = blockIdx.x / HQ, hq = blockIdx.x - u * HQ, h = hq / maps, t = row0 ? row0[u] : u;
  const size_t rec = (size_t)Vp + 4;
  const float v = merge_splits(ws + ((size_t)t * HQ + hq) * rec, (size_t)rows_total * rec, nsplit, Vp, DV, wgt, red);
  if (threadIdx.x < DV) st_any(out, (size_t)t * ldo + (size_t)hq * DV + threadIdx.x, odt, v * (gate ? gate[(size_t)t * ldg + h] : 1.f));
}

// one workgroup per (row, head) of two maps: both merged, then d = first - lam * second, y = d / sqrt(mean(d^2) + eps) * out_scale
__global__ __launch_bounds__(256) void gqa_attn_merge_diff_kernel(void* __restrict__ y, int ydt, long ldy, const float* __restrict__ ws, int nsplit,
                                                                  int rows_total, int H, int DV, int Vp, const float* __restrict__ gate, long ldg,
                                                                  float lam, float out_scale, float eps) {
  __shared__ float wgt[1024];
  __shared__ float red[4];
  const int gi = blockIdx.x, t = gi / H, h = gi - t * H;
  const size_t rec = (size_t)Vp + 4, stride = (size_t)rows_total * rec;
  const float* base = ws + ((size_t)t * H * 2 + (size_t)h * 2) * rec;
  const float a1 = merge_splits(base, stride, nsplit, Vp, DV, wgt, red);
  const float a2 = merge_splits(base + rec, stride, nsplit, Vp, DV, wgt, red);
  const float d = (a1 - lam * a2) * (gate ? gate[(size_t)t * ldg + h] : 1.f);
  const float inv = out_scale / sqrtf(block256_sum(d * d, red) / (float)DV + eps);
  if (threadIdx.x < DV) st_any(y, (size_t)t * ldy + (size_t)h * DV + threadIdx.x, ydt, d * inv);
}

// One token of each request (decoding), from the rows of the input product to those of the output product: norm, rotation and append of prep, attention, and the merge of
// the waves.  In three launches (prep, tile kernel in splits, merge) each waits for its own chain of slot, page and data, and of a tile kernel's four waves three had no row: a
// workgroup owns a (request, key head), and its waves take 64-key tiles in turn, each with slots of LDS, a softmax and sums of its own, which meet in LDS at the end.
//   * a wave asks for its next tile's keys behind the reads of this one's, for the values likewise: only the wave itself waits for its loads;
//   * the token's own key and value are made by the wave whose tile holds their position, put over that tile's row in LDS (the page's is stale) and, behind the walk, into the page;
//   * walks too long for a workgroup are split as the tile kernel's are (gqa_attn_merge_kernel adds them).
// Bound by the chain of launch, slot, page pointer and tiles, and past that by one workgroup's LDS in flight (128 KB a unit): 32 heads over 8 of 128, one launch against three, in us
// (keys: 100 / 700 / 1500 / 4000 / 12000): 1 request 8.0 / 11.0 / 11.1 / 13.1 / 18.1 (13.3 / 13.6 / 14.2 / 18.7 / 22.4), 4 requests 8.1 / 12.7 / 14.3 / 18.5 / 41.5 (13.5 / 16.3 / 18.3 /
// 23.1 / 48.4), 32 requests 9.8 / 22.5 / 41.7 / 94.0 (17.5 / 31.2 / 52.0 / 110).
template <int D, int DV, bool CAP>
__global__ __launch_bounds__(256) void gqa_decode_step_kernel(PrepArgs p, GqaArgs a) {
  constexpr int KS = D / 32, DT = DV / 16, NT = 4, WAVES = 4;
  constexpr int KROW = D * 2, VROW = DV * 2, KBYTES = 64 * KROW, VBYTES = 64 * VROW, SLOT = KBYTES + VBYTES;
  constexpr int KPP = 1024 / KROW, VPP = 1024 / VROW, KP = 64 / KPP, VP = 64 / VPP;   // keys per 1 KiB piece, pieces of a tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // [wave][keys | values]; at the end [wave][16 heads][DV + 4] f32
  __shared__ float cs_t[64], sn_t[64];
  const int H = a.H, G = a.G, hpg = H / G, e = blockIdx.x / G, g = blockIdx.x - e * G, split = blockIdx.y, nsplit = gridDim.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ni = lane & 15, kb = lane >> 4;
  const int row0 = a.ent_row0[e];
  void* const* gkp = a.kspans + (size_t)a.ent_slot[e] * a.span_stride;
  void* const* gvp = a.vspans + (size_t)a.ent_slot[e] * a.span_stride;
  const int first = split * WAVES + wave, stride = WAVES * nsplit;   // the wave's tiles: first + i * stride
  const float* row = p.qkv + (size_t)row0 * p.ld;
  // the wave's page pointers, 64 tiles at a time, one to a lane (a table row's entries past the request's pages are not followed)
  const int tpp = a.span_len >> 6, room = a.span_stride * tpp;       // tiles per page, of a table row
  uint64_t kptr = 0, vptr = 0;
  auto pages = [&](int i0) {
    const int t = first + stride * (i0 + lane);
    if (t < room) {
      kptr = (uint64_t)gload<void*>(gkp + t / tpp);
      vptr = (uint64_t)gload<void*>(gvp + t / tpp);
    }
  };
  auto tiles = [&](int i0) {         // .. from the page to the tile (apart: the loads are not waited for where they are asked for)
    const int t = first + stride * (i0 + lane);
    kptr += (size_t)(t % tpp) * 64 * G * KROW;
    vptr += (size_t)(t % tpp) * 64 * G * VROW;
  };
  // where this lane's 16 bytes of pieces q, q + 4, .. come from (the chunks of a row change places as in the tile kernel)
  const int kk = lane / (KROW / 16), kc = lane % (KROW / 16), vk = lane / (VROW / 16), vc = lane % (VROW / 16);
  uint32_t koff[4], voff[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int key = q * KPP + kk, val = q * VPP + vk;
    koff[q] = (uint32_t)(key * G + g) * KROW + (uint32_t)((kc ^ (D == 128 ? key & 15 : key & 7)) * 16);
    voff[q] = (uint32_t)(val * G + g) * VROW + (uint32_t)((vc ^ (DV == 128 ? (val & 7) * 2 : ((val >> 1) & 3) * 2)) * 16);
  }
  unsigned char* const kbuf = smem + wave * SLOT;
  unsigned char* const vbuf = kbuf + KBYTES;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * SLOT;
  auto lane_ptr = [&](uint64_t ptr, int i) {
    return (const char*)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)ptr, i) | (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(ptr >> 32), i) << 32);
  };
  auto fetch_k = [&](int i) {
    const char* from = lane_ptr(kptr, i & 63);
#pragma unroll
    for (int j = 0; j < KP; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + j * 1024), "v"(koff[j & 3]), "s"(from + (size_t)(j >> 2) * 4 * KPP * G * KROW) : "memory");
  };
  auto fetch_v = [&](int i) {
    const char* from = lane_ptr(vptr, i & 63);
#pragma unroll
    for (int j = 0; j < VP; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + KBYTES + j * 1024), "v"(voff[j & 3]), "s"(from + (size_t)(j >> 2) * 4 * VPP * G * VROW) : "memory");
  };
  // what the prologue reads, beside the page pointers and in front of the tiles (loads return in order: behind them it would wait for all of them): the query row of the
  // lane's head, the token's key and value (D / 64, DV / 64 neighbours to a lane), the norms' weights
  constexpr int KE = D / 64, VE = DV / 64;
  const int h = g * hpg + min(ni, hpg - 1), half = p.rot_dims >> 1;
  const float* qrow = row + p.q_off + (size_t)h * D + kb * 8;
  pages(0);
  f32x4_t qv[KS][2], qw[KS][2];
  float kn[KE], kw[KE], vn[VE];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qv[ks][0] = *reinterpret_cast<const f32x4_t*>(qrow + ks * 32);
    qv[ks][1] = *reinterpret_cast<const f32x4_t*>(qrow + ks * 32 + 4);
  }
#pragma unroll
  for (int i = 0; i < KE; ++i) kn[i] = row[p.k_off + (size_t)g * D + lane * KE + i];
#pragma unroll
  for (int i = 0; i < VE; ++i) vn[i] = row[p.v_off + (size_t)g * DV + lane * VE + i];
  int pos = a.tok_pos[row0];
  asm volatile("" : "+s"(pos));      // (asked for here, not where it is used)
  const int last = pos >> 6, mine = last >= first ? (last - first) / stride + 1 : 0;
  const bool owner = mine > 0 && (last - first) % stride == 0;       // (uniform) the wave's last tile holds the token
  // (one branch on the weights' type around all of them, what is not there read from the row instead and not used: a branch for each would wait for each)
  constexpr float LOG2E = 1.44269504088896341f;
  const void* const qnp = p.qnorm ? p.qnorm : row;
  const void* const knp = p.knorm ? p.knorm : row;
  const bool w32 = p.wdt == DIHIP_F32;
  uint32_t qb[KS * 8], kbits[KE];
  if (w32) {
#pragma unroll
    for (int x = 0; x < KS * 8; ++x) qb[x] = ((const uint32_t*)qnp)[(x >> 3) * 32 + kb * 8 + (x & 7)];
#pragma unroll
    for (int i = 0; i < KE; ++i) kbits[i] = ((const uint32_t*)knp)[lane * KE + i];
  } else {
#pragma unroll
    for (int x = 0; x < KS * 8; ++x) qb[x] = (uint32_t)((const uint16_t*)qnp)[(x >> 3) * 32 + kb * 8 + (x & 7)] << 16;
#pragma unroll
    for (int i = 0; i < KE; ++i) kbits[i] = (uint32_t)((const uint16_t*)knp)[lane * KE + i] << 16;
  }
  const bool with_sink = a.sink_mode != 0 && split == 0 && wave == 0;
  float fr = tid < half ? p.freq[tid] : 0.f;
  float m = with_sink ? (a.sink_mode == 1 ? ld_any(a.sink, h, a.wdt) * LOG2E : 0.f) : -1e30f, l = with_sink && kb == 0 ? 1.f : 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {   // all of it is here
    asm volatile("" : "+v"(qv[ks][0]), "+v"(qv[ks][1]));
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      qw[ks][x >> 2][x & 3] = p.qnorm ? __builtin_bit_cast(float, qb[ks * 8 + x]) : 1.f;
    }
    asm volatile("" : "+v"(qw[ks][0]), "+v"(qw[ks][1]));
  }
#pragma unroll
  for (int i = 0; i < KE; ++i) {
    kw[i] = p.knorm ? __builtin_bit_cast(float, kbits[i]) : 1.f;
    asm volatile("" : "+v"(kn[i]), "+v"(kw[i]));
  }
#pragma unroll
  for (int i = 0; i < VE; ++i) asm volatile("" : "+v"(vn[i]));
  asm volatile("" : "+v"(m), "+v"(fr), "+v"(kptr), "+v"(vptr));
  tiles(0);
  if (mine > 0) {
    fetch_k(0);
    fetch_v(0);
  }
  if (tid < half) {
    float sn, cs;
    rope_sincos((uint32_t)pos, fr, &sn, &cs);
    cs_t[tid] = cs * p.mag;
    sn_t[tid] = sn * p.mag;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (not __syncthreads: it would wait for the tiles)
  u32x4_t qf[KS];
  {
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) ss = __builtin_fmaf(qv[ks][c][r], qv[ks][c][r], ss);
    if (p.qnorm) {
      const float inv = 1.f / sqrtf(rows_sum(ss) / (float)D + p.eps);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) qv[ks][c][r] = qv[ks][c][r] * inv * qw[ks][c][r];
    }
    if (half) {    // (rot_dims == D)
      if (p.layout == 0) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
              const int pair = (ks * 32 + kb * 8 + c * 4 + r) >> 1;
              const float x = qv[ks][c][r], y = qv[ks][c][r + 1], cs = cs_t[pair], sn = sn_t[pair];
              qv[ks][c][r] = x * cs - y * sn;
              qv[ks][c][r + 1] = y * cs + x * sn;
            }
      } else {
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int pair = ks * 32 + kb * 8 + c * 4 + r;
              const float x = qv[ks][c][r], y = qv[ks + KS / 2][c][r], cs = cs_t[pair], sn = sn_t[pair];
              qv[ks][c][r] = x * cs - y * sn;
              qv[ks + KS / 2][c][r] = y * cs + x * sn;
            }
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = u32x4_t{pack_bf16x2(qv[ks][0][0], qv[ks][0][1]), pack_bf16x2(qv[ks][0][2], qv[ks][0][3]), pack_bf16x2(qv[ks][1][0], qv[ks][1][1]), pack_bf16x2(qv[ks][1][2], qv[ks][1][3])};
  }
  if (owner) {   // the token's key: norm, rotation
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < KE; ++i) ss = __builtin_fmaf(kn[i], kn[i], ss);
    if (p.knorm) {
      const float inv = 1.f / sqrtf(wave_sum(ss) / (float)D + p.eps);
#pragma unroll
      for (int i = 0; i < KE; ++i) kn[i] = kn[i] * inv * kw[i];
    }
    if (half) {
      float other[KE];
#pragma unroll
      for (int i = 0; i < KE; ++i) other[i] = p.layout == 1 ? __shfl_xor(kn[i], 32, 64) : KE == 2 ? kn[KE - 1 - i] : __shfl_xor(kn[i], 1, 64);
#pragma unroll
      for (int i = 0; i < KE; ++i) {
        const int d = lane * KE + i;
        const bool low = p.layout == 1 ? d < half : (d & 1) == 0;
        const int pair = p.layout == 1 ? (d < half ? d : d - half) : d >> 1;
        kn[i] = low ? kn[i] * cs_t[pair] - other[i] * sn_t[pair] : kn[i] * cs_t[pair] + other[i] * sn_t[pair];
      }
    }
  }
  f32x4_t oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) oacc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int kfo[KS], vfo[DT];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kfo[ks] = ni * KROW + (((ks * 4 + kb) ^ (D == 128 ? ni : ni & 7)) * 16);
  {
    const int vr = kb * 4 + (ni >> 2), f = DV == 128 ? (vr & 7) * 2 : ((vr >> 1) & 3) * 2;
#pragma unroll
    for (int t = 0; t < DT; ++t) vfo[t] = vr * VROW + (((2 * t) ^ f) + ((ni & 3) >> 1)) * 16 + (ni & 1) * 8;
  }
  const float sl2 = a.scale * LOG2E, cap = a.softcap, cap_in = CAP ? 2.f * a.scale * LOG2E / cap : 0.f, cap2 = cap * LOG2E;
  for (int i = 0; i < mine; ++i) {
    const int key0 = (first + stride * i) * 64;
    const bool here = owner && i + 1 == mine;        // (uniform) the tile of the token, and of rows that no token has written
    // keys: everything but the values' pieces behind them has landed
    if (here) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VP) : "memory");
    const int r = pos & 63;
    if (here) {
      const int d = lane * KE;
      unsigned char* to = kbuf + r * KROW + ((d >> 3) ^ (D == 128 ? r & 15 : r & 7)) * 16 + (d & 7) * 2;
      if constexpr (KE == 2) *reinterpret_cast<uint32_t*>(to) = pack_bf16x2(kn[0], kn[1]);
      else *reinterpret_cast<uint16_t*>(to) = (uint16_t)f32_to_bf16_bits(kn[0]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    f32x4_t sacc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sacc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4_t kf[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) kf[nt] = *reinterpret_cast<const u32x4_t*>(kbuf + kfo[ks] + nt * 16 * KROW);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) sacc[nt] = mfma_bf16g(kf[nt], qf[ks], sacc[nt]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the keys have been read
    const bool more = i + 1 < mine;
    if (more) {
      if (((i + 1) & 63) == 0) {
        pages(i + 1);
        tiles(i + 1);
      }
      fetch_k(i + 1);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float x;
        if constexpr (CAP) x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(sacc[nt][q] * cap_in));   // cap * tanh(s / cap)
        else x = sacc[nt][q] * sl2;
        if (here && key0 + nt * 16 + kb * 4 + q > pos) x = -INFINITY;
        sacc[nt][q] = x;
        mx = fmaxf(mx, x);
      }
    mx = fmaxf(m, rows_max(mx));
    const float corr = __builtin_amdgcn_exp2f(m - mx);
    m = mx;
    float ps = 0.f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sacc[nt][q] = __builtin_amdgcn_exp2f(sacc[nt][q] - mx);
        ps += sacc[nt][q];
      }
    l = l * corr + ps;
    u32x4_t pf[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
      pf[hh] = u32x4_t{pack_bf16x2(sacc[2 * hh][0], sacc[2 * hh][1]), pack_bf16x2(sacc[2 * hh][2], sacc[2 * hh][3]),
                       pack_bf16x2(sacc[2 * hh + 1][0], sacc[2 * hh + 1][1]), pack_bf16x2(sacc[2 * hh + 1][2], sacc[2 * hh + 1][3])};
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) oacc[t][q] *= corr;
    // values: this tile's have landed, the next one's keys may be on their way
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(KP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (here) {
      const int d = lane * VE;
      unsigned char* to = vbuf + r * VROW + ((d >> 3) ^ (DV == 128 ? (r & 7) * 2 : ((r >> 1) & 3) * 2)) * 16 + (d & 7) * 2;
      if constexpr (VE == 2) *reinterpret_cast<uint32_t*>(to) = pack_bf16x2(vn[0], vn[1]);
      else *reinterpret_cast<uint16_t*>(to) = (uint16_t)f32_to_bf16_bits(vn[0]);
      for (int z = lane; z < (63 - r) * (VROW / 16); z += 64) *reinterpret_cast<u32x4_t*>(vbuf + (r + 1) * VROW + z * 16) = u32x4_t{0u, 0u, 0u, 0u};   // (an infinity there, times 0)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const u32x2_t lo2 = lds_read_tr16(vbuf + vfo[t] + hh * 32 * VROW), hi2 = lds_read_tr16(vbuf + vfo[t] + hh * 32 * VROW + 16 * VROW);
        const u32x4_t vf = {lo2[0], lo2[1], hi2[0], hi2[1]};
        oacc[t] = mfma_bf16g(vf, pf[hh], oacc[t]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the values have been read
    if (more) fetch_v(i + 1);
  }
  if (owner) {   // the token's key and value into their page, off the way of the tiles
    const int i = (mine - 1) & 63, r = pos & 63;
    uint16_t* kto = (uint16_t*)(lane_ptr(kptr, i) + (size_t)(r * G + g) * KROW) + lane * KE;
    uint16_t* vto = (uint16_t*)(lane_ptr(vptr, i) + (size_t)(r * G + g) * VROW) + lane * VE;
#pragma unroll
    for (int x = 0; x < KE; ++x) kto[x] = (uint16_t)f32_to_bf16_bits(kn[x]);
#pragma unroll
    for (int x = 0; x < VE; ++x) vto[x] = (uint16_t)f32_to_bf16_bits(vn[x]);
  }
  l = rows_sum(l);
  __syncthreads();     // every wave has read its last tile (and waited for its last load): the sums meet in their place
  float* const rec = reinterpret_cast<float*>(smem);
  if (ni < hpg) {
    float* o = rec + (size_t)(wave * 16 + ni) * (DV + 4);
#pragma unroll
    for (int t = 0; t < DT; ++t) *reinterpret_cast<f32x4_t*>(o + t * 16 + kb * 4) = oacc[t];
    if (kb == 0) {
      o[DV] = m;
      o[DV + 1] = l;
    }
  }
  __syncthreads();
  for (int x = tid; x < hpg * (DV / 4); x += 256) {
    const int hh = x / (DV / 4), d = (x - hh * (DV / 4)) * 4;
    float mw[WAVES], M = -1e30f, den = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      mw[w] = rec[(w * 16 + hh) * (DV + 4) + DV];
      M = fmaxf(M, mw[w]);
    }
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float c = __builtin_amdgcn_exp2f(mw[w] - M);
      const float* from = rec + (w * 16 + hh) * (DV + 4);
      den = __builtin_fmaf(c, from[DV + 1], den);
      o += c * *reinterpret_cast<const f32x4_t*>(from + d);
    }
    const int head = g * hpg + hh;
    if (nsplit == 1) {
      const float inv = (a.gate ? a.gate[(size_t)row0 * a.ldg + head] : 1.f) / den;
      store4(a.out, (size_t)row0 * a.ldo + (size_t)head * DV + d, a.odt, o * inv);
    } else {   // [split][row, query head][DV sums, maximum, denominator, ..]
      float* to = a.ws + ((size_t)split * a.rows_total + (size_t)row0 * H + head) * (DV + 4);
      *reinterpret_cast<f32x4_t*>(to + d) = o;
      if (d == 0) {
        to[DV] = M * 0.69314718055994531f;
        to[DV + 1] = den;
      }
    }
  }
}

}  // namespace
}  // namespace dihip

using namespace dihip;

extern "C" {

int dihip_qkv_prep_append(void* stream, float* qkv, long ld, int q_off, int k_off, int v_off, int H, int G, int D, int DV, int maps,
                          const void* qnorm, const void* knorm, int w_dtype, float eps, const float* freq, int rot_dims, int layout,
                          float mag, float lam, const float* vfirst_in, float* vfirst_out, long ldvf, void* const* kspans,
                          void* const* vspans, int span_stride, int span_len, int cache_dtype, const int32_t* tok_slot,
                          const int32_t* tok_pos, int T) {
  DIHIP_REQUIRE(T >= 0 && qkv && H > 0 && G > 0 && H % G == 0 && D > 0 && D <= 256 && DV > 0 && kspans && vspans && tok_slot && tok_pos &&
                    span_stride > 0 && span_len > 0 && seq_dtype_ok(cache_dtype) && seq_dtype_ok(w_dtype), DIHIP_PARAM_ERROR,
                "qkv_prep_append: bad argument (heads of at most 256 elements)");
  DIHIP_REQUIRE(maps >= 1 && maps <= 8, DIHIP_PARAM_ERROR, "qkv_prep_append: 1 to 8 maps per head");
  const int GV = G;
  H *= maps;     // from here on: query / key vectors per token
  G *= maps;
  DIHIP_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && ld >= (long)q_off + (long)H * D && ld >= (long)k_off + (long)G * D &&
                    ld >= (long)v_off + (long)GV * DV, DIHIP_PARAM_ERROR, "qkv_prep_append: columns outside the rows");
  DIHIP_REQUIRE(rot_dims >= 0 && rot_dims <= D && rot_dims % 2 == 0 && (rot_dims == 0 || freq) && (layout == 0 || layout == 1),
                DIHIP_PARAM_ERROR, "qkv_prep_append: bad rotation (an even number of dimensions up to the head size, layout 0 / 1)");
  DIHIP_REQUIRE((!vfirst_in && !vfirst_out) || ldvf >= (long)GV * DV, DIHIP_PARAM_ERROR, "qkv_prep_append: value rows shorter than the values");
  if (T == 0) return DIHIP_SUCCESS;
  PrepArgs a{qkv, ld, q_off, k_off, v_off, H, G, D, DV, GV, qnorm, knorm, w_dtype, eps, freq, rot_dims, layout, mag, lam, vfirst_in, vfirst_out,
             ldvf, kspans, vspans, span_stride, span_len, cache_dtype, tok_slot, tok_pos};
  const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if ((D == 64 || D == 128) && rot_dims % 8 == 0 && cache_dtype == DIHIP_BF16 && (GV * DV) % 4 == 0 && al16(qkv) && ((ld | q_off | k_off | v_off) & 3) == 0 &&
      al16(vfirst_in) && al16(vfirst_out) && ((!vfirst_in && !vfirst_out) || ldvf % 4 == 0)) {
    // few rows (decoding): a token's heads one to a lane group; many rows: a workgroup per token
    const int per = 4 * 64 / (D / 4), gy = T >= 256 ? 1 : (H + G + per - 1) / per;
    const auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(T, gy), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), a); };
    if (D == 64) gy > 1 || per >= H + G ? go(qkv_prep_append_vec_kernel<64, 1>) : go(qkv_prep_append_vec_kernel<64, 4>);
    else gy > 1 || per >= H + G ? go(qkv_prep_append_vec_kernel<128, 1>) : go(qkv_prep_append_vec_kernel<128, 4>);
    return launch_status();
  }
  // few rows (decoding): the heads of a token are spread over workgroups of four; many rows: a workgroup per token
  hipLaunchKernelGGL(qkv_prep_append_kernel, dim3(T, T >= 256 ? 1 : (H + G + 3) / 4), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), a);
  return launch_status();
}

int dihip_qkv_conv_prep_append(void* stream, const float* x, long ld, const void* conv, int taps, float* tail, int write_tail, int H, int G, int D,
                               int DV, const void* qnorm, const void* knorm, int w_dtype, float eps, const float* freq, int rot_dims, int layout,
                               float mag, float* q_out, long ldq, void* const* kspans, void* const* vspans, int span_stride, int span_len,
                               int cache_dtype, const int32_t* tok_slot, const int32_t* tok_pos, const int32_t* tok_off, int T) {
  DIHIP_REQUIRE(T >= 0 && x && conv && H > 0 && G > 0 && H % G == 0 && D > 0 && DV > 0 && q_out && kspans && vspans && tok_slot && tok_pos && tok_off &&
                    span_stride > 0 && span_len > 0 && seq_dtype_ok(cache_dtype) && seq_dtype_ok(w_dtype), DIHIP_PARAM_ERROR,
                "qkv_conv_prep_append: bad argument");
  DIHIP_REQUIRE(taps >= 1 && taps <= 16 && (tail || taps == 1), DIHIP_PARAM_ERROR, "qkv_conv_prep_append: 1 to 16 taps, with their state");
  DIHIP_REQUIRE(ld >= (long)(H + G) * D + (long)G * DV && ldq >= (long)H * D, DIHIP_PARAM_ERROR, "qkv_conv_prep_append: columns outside the rows");
  DIHIP_REQUIRE(rot_dims >= 0 && rot_dims <= D && rot_dims <= 256 && rot_dims % 2 == 0 && (rot_dims == 0 || freq) && (layout == 0 || layout == 1),
                DIHIP_PARAM_ERROR, "qkv_conv_prep_append: bad rotation (an even number of at most 256 dimensions up to the head size, layout 0 / 1)");
  DIHIP_REQUIRE((long)H * D <= 15360, DIHIP_EXCEED_LIMIT_ERROR, "qkv_conv_prep_append: query rows of more than 15360 elements");
  if (T == 0) return DIHIP_SUCCESS;
  ConvPrepArgs a{x, ld, conv, qnorm, knorm, w_dtype, taps, taps > 1 ? tail : nullptr, write_tail && taps > 1, eps, freq, rot_dims, layout == 0, mag, q_out, ldq,
                 kspans, vspans, span_stride, span_len, cache_dtype, tok_slot, tok_pos, tok_off, H * D, G * D, G * DV, D};
  const size_t lds = (size_t)H * D * sizeof(float);      // (G <= H: the key row fits too)
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  const int C = (H + G) * D + G * DV, longest = H * D > G * DV ? H * D : G * DV;
  if (D % 4 == 0 && DV % 4 == 0 && al16(x) && ld % 4 == 0 && al16(conv) && (!a.tail || al16(tail)) && al16(q_out) && ldq % 4 == 0 && (!qnorm || al16(qnorm)) &&
      (!knorm || al16(knorm)) && C % 4 == 0 && longest <= 16384) {
    auto go = [&](auto wt, auto nt, auto ept) {
      constexpr int WT = decltype(wt)::value, NT = decltype(nt)::value, EPT = decltype(ept)::value;
      hipLaunchKernelGGL((qkv_conv_prep_append_vec_kernel<WT, NT, EPT>), dim3(T, 3), dim3(NT), layout == 1 && rot_dims ? lds : 0, s, a);
    };
    auto by_n = [&](auto wt) {
      using one = std::integral_constant<int, 1>;
      if (longest <= 1024) go(wt, std::integral_constant<int, 256>{}, one{});
      else if (longest <= 2048) go(wt, std::integral_constant<int, 512>{}, one{});
      else if (longest <= 4096) go(wt, std::integral_constant<int, 1024>{}, one{});
      else if (longest <= 8192) go(wt, std::integral_constant<int, 1024>{}, std::integral_constant<int, 2>{});
      else go(wt, std::integral_constant<int, 1024>{}, std::integral_constant<int, 4>{});
    };
    if (w_dtype == DIHIP_F32) by_n(std::integral_constant<int, DIHIP_F32>{});
    else by_n(std::integral_constant<int, DIHIP_BF16>{});
    return launch_status();
  }
  if (H * D <= 1024) hipLaunchKernelGGL(qkv_conv_prep_append_kernel<256>, dim3(T, 3), dim3(256), lds, s, a);
  else hipLaunchKernelGGL(qkv_conv_prep_append_kernel<1024>, dim3(T, 3), dim3(1024), lds, s, a);
  return launch_status();
}

static int gqa_check(const char* what, const void* out, int odt, long ldo, const float* q, long ldq, void* const* kspans, void* const* vspans,
                     int span_stride, int span_len, const void* sink, int w_dtype, int sink_mode, const float* gate, long ldg, int H, int G,
                     int D, int DV, int maps, int keep_first) {
  DIHIP_REQUIRE(maps >= 1 && maps <= 8 && keep_first >= 0, DIHIP_PARAM_ERROR, "%s: 1 to 8 maps per head, no negative count of kept keys", what);
  DIHIP_REQUIRE(out && q && kspans && vspans && span_stride > 0 && span_len > 0 && H > 0 && G > 0 && H % G == 0 && D > 0 && DV > 0 &&
                    ldo >= (long)H * maps * DV && ldq >= (long)H * maps * D && seq_dtype_ok(w_dtype) && seq_dtype_ok(odt), DIHIP_PARAM_ERROR, "%s: bad argument", what);
  DIHIP_REQUIRE(sink_mode >= 0 && sink_mode <= 2 && (sink_mode != 1 || sink) && (!gate || ldg >= H || ldg == 0), DIHIP_PARAM_ERROR,
                "%s: bad sink mode or gate", what);
  return DIHIP_SUCCESS;
}

int dihip_gqa_attn(void* stream, void* out, int out_dtype, long ldo, const float* q, long ldq, void* const* kspans, void* const* vspans,
                   int span_stride, int span_len, int cache_dtype, const void* sink, int w_dtype, int sink_mode, float softcap,
                   const float* gate, long ldg, const int32_t* tok_slot, const int32_t* tok_pos, int T, int H, int G, int D, int DV,
                   float scale, int maps, int window, int keep_first) {
  if (int rc = gqa_check("gqa_attn", out, out_dtype, ldo, q, ldq, kspans, vspans, span_stride, span_len, sink, w_dtype, sink_mode, gate, ldg, H, G, D, DV, maps, keep_first)) return rc;
  DIHIP_REQUIRE(T >= 0 && tok_slot && tok_pos && seq_dtype_ok(cache_dtype), DIHIP_PARAM_ERROR, "gqa_attn: bad argument");
  DIHIP_REQUIRE(D <= 256 && DV <= 512, DIHIP_EXCEED_LIMIT_ERROR, "gqa_attn: head sizes above 256 (keys) / 512 (values)");
  if (T == 0) return DIHIP_SUCCESS;
  GqaArgs a{out, out_dtype, ldo, q, ldq, kspans, vspans, span_stride, span_len, sink, w_dtype, sink_mode, softcap, gate, ldg, tok_slot, tok_pos,
            nullptr, nullptr, nullptr, H, G, D, DV, scale, nullptr, 0, maps, window, keep_first};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto go = [&](auto ct, auto rv) {
    constexpr int CT = decltype(ct)::value, RV = decltype(rv)::value;
    hipLaunchKernelGGL((gqa_attn_kernel<CT, RV>), dim3(T), dim3(256), 0, s, a);
  };
  auto by_v = [&](auto ct) {
    if (DV <= 64) go(ct, std::integral_constant<int, 1>{});
    else if (DV <= 128) go(ct, std::integral_constant<int, 2>{});
    else if (DV <= 256) go(ct, std::integral_constant<int, 4>{});
    else go(ct, std::integral_constant<int, 8>{});
  };
  if (cache_dtype == DIHIP_F32) by_v(std::integral_constant<int, DIHIP_F32>{});
  else by_v(std::integral_constant<int, DIHIP_BF16>{});
  return launch_status();
}

int dihip_gqa_attn_mc_supported(int D, int DV, int span_len, int cache_dtype) {
  return cache_dtype == DIHIP_BF16 && D % 8 == 0 && DV % 8 == 0 && D >= 8 && DV >= 8 && D <= 256 && DV <= 128 && span_len % 32 == 0;
}

size_t dihip_gqa_attn_mc_workspace_bytes(int T, int HQ, int DV, int nsplit) {
  return nsplit > 1 ? (size_t)nsplit * T * HQ * (((DV + 15) & ~15) + 4) * sizeof(float) : 0;
}

int dihip_gqa_attn_mc(void* stream, void* out, int out_dtype, long ldo, const float* q, long ldq, void* const* kspans, void* const* vspans,
                      int span_stride, int span_len, const void* sink, int w_dtype, int sink_mode, float softcap, const float* gate,
                      long ldg, const int32_t* tok_pos, const int32_t* ent_slot, const int32_t* ent_row0, const int32_t* ent_count, int E,
                      int max_count, int T, int H, int G, int D, int DV, float scale, int maps, int window, int keep_first, int nsplit,
                      void* ws, size_t ws_bytes, void* diff_out, int diff_dtype, long ldd, float lam, float out_scale, float eps) {
  if (int rc = gqa_check("gqa_attn_mc", out, out_dtype, ldo, q, ldq, kspans, vspans, span_stride, span_len, sink, w_dtype, sink_mode, gate, ldg, H, G, D, DV, maps, keep_first)) return rc;
  DIHIP_REQUIRE(dihip_gqa_attn_mc_supported(D, DV, span_len, DIHIP_BF16), DIHIP_PARAM_ERROR,
                "gqa_attn_mc: head sizes %d / %d (multiples of 8 up to 256 / 128) or span_len %d (a multiple of 32) not served", D, DV, span_len);
  DIHIP_REQUIRE(E >= 0 && T >= 0 && max_count >= 0 && tok_pos && ent_slot && ent_row0 && ent_count && ldo % 4 == 0 && ldq % 4 == 0,
                DIHIP_PARAM_ERROR, "gqa_attn_mc: bad argument");
  DIHIP_REQUIRE((reinterpret_cast<uintptr_t>(out) & 15u) == 0 && (reinterpret_cast<uintptr_t>(q) & 15u) == 0, DIHIP_PARAM_ERROR,
                "gqa_attn_mc: q / out must be 16-byte aligned");
  DIHIP_REQUIRE(nsplit >= 1 && nsplit <= 1024 && (long)E * G * maps <= 65535, DIHIP_PARAM_ERROR, "gqa_attn_mc: bad split / portion count");
  DIHIP_REQUIRE(!diff_out || (maps == 2 && out_dtype == DIHIP_F32 && ldd >= (long)H * DV && seq_dtype_ok(diff_dtype)), DIHIP_PARAM_ERROR,
                "gqa_attn_mc: the difference of the maps needs two maps and rows of H * DV elements");
  DIHIP_REQUIRE(ws_bytes >= dihip_gqa_attn_mc_workspace_bytes(T, H * maps, DV, nsplit) && (nsplit == 1 || ws), DIHIP_PARAM_ERROR,
                "gqa_attn_mc: workspace too small");
  if (E == 0 || max_count == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  GqaArgs a{out, out_dtype, ldo, q, ldq, kspans, vspans, span_stride, span_len, sink, w_dtype, sink_mode, softcap, gate, ldg, nullptr, tok_pos,
            ent_slot, ent_row0, ent_count, H, G, D, DV, scale, (float*)ws, T * H * maps, maps, window, keep_first};
  const int hpg = H / G, Dp = (D + 31) & ~31, Vp = (DV + 15) & ~15;
  const dim3 grid((unsigned)(((long)max_count * hpg + 63) / 64), E * G * maps, nsplit);
  const size_t lds = (size_t)32 * ((Dp + 8) + (Vp + 8)) * 2;
  auto go = [&](auto dm, auto vm) {
    constexpr int DM = decltype(dm)::value, VM = decltype(vm)::value;
    hipLaunchKernelGGL((gqa_attn_mc_kernel<DM, VM>), grid, dim3(256), lds, s, a);
  };
  auto by_v = [&](auto dm) {
    if (DV <= 64) go(dm, std::integral_constant<int, 64>{});
    else go(dm, std::integral_constant<int, 128>{});
  };
  // head sizes of exactly 64 / 128, whole 64-key tiles per page
  const bool tiles = (D == 64 || D == 128) && (DV == 64 || DV == 128) && span_len % 64 == 0;
  auto go_tile = [&](auto d, auto v, auto mt, auto cap) {
    constexpr int D_ = decltype(d)::value, V_ = decltype(v)::value, MT = decltype(mt)::value;
    constexpr bool CAP = decltype(cap)::value;
    const int gx = (int)(((long)max_count * hpg + 64 * MT - 1) / (64 * MT));
    const size_t bytes = (size_t)2 * 64 * (D_ + V_) * 2;
    auto kern = gqa_attn_tile_kernel<D_, V_, MT, CAP>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return;   // (reported below)
    hipLaunchKernelGGL(kern, dim3((unsigned)gx * E * G * maps, 1, nsplit), dim3(256), bytes, s, a, gx);
  };
  auto by_cap = [&](auto d, auto v, auto mt) {
    if (softcap > 0.f) go_tile(d, v, mt, std::true_type{});
    else go_tile(d, v, mt, std::false_type{});
  };
  auto by_mt = [&](auto d, auto v) {
    // two 16-pair operands per wave where that still gives most CUs the two workgroups they hold.  One operand / two, us: 32 heads over 8, 1000 rows behind 1000
    // (256 workgroups of two operands) 55 / 73, 16 over 16 3000 rows (384) 67 / 91, 32 over 8 two portions of 500 rows that see 16 keys (256) 13.7 / 17.0; but 64 over 4 1000 rows
    // behind 1000 (500) 91 / 82, 32 over 8 3000 rows (752) 125 / 107
    const long most = ((long)max_count * hpg + 127) / 128 * E, held = (long)T * hpg / 128 + E;   // row tiles: by the longest portion, by all rows
    if ((long)max_count * hpg > 64 && std::min(most, held) * G * maps * nsplit >= 448) by_cap(d, v, std::integral_constant<int, 2>{});
    else by_cap(d, v, std::integral_constant<int, 1>{});
  };
  constexpr std::integral_constant<int, 64> c64{};
  constexpr std::integral_constant<int, 128> c128{};
  if (tiles) {
    if (D == 64 && DV == 64) by_mt(c64, c64);
    else if (D == 64) by_mt(c64, c128);
    else if (DV == 64) by_mt(c128, c64);
    else by_mt(c128, c128);
  } else if (D <= 64) by_v(std::integral_constant<int, 64>{});
  else if (D <= 128) by_v(std::integral_constant<int, 128>{});
  else by_v(std::integral_constant<int, 256>{});
  if (nsplit > 1 && diff_out)      // the merge of both maps, their difference and its norm in one launch
    hipLaunchKernelGGL(gqa_attn_merge_diff_kernel, dim3(T * H), dim3(256), 0, s, diff_out, diff_dtype, ldd, (const float*)ws, nsplit, T * H * maps, H, DV,
                       Vp, gate, ldg, lam, out_scale, eps);
  else if (nsplit > 1)
    hipLaunchKernelGGL(gqa_attn_merge_kernel, dim3(T * H * maps), dim3(256), 0, s, out, out_dtype, ldo, (const float*)ws, nsplit, T * H * maps, H, maps, DV, Vp, gate, ldg,
                       (const int32_t*)nullptr);
  else if (diff_out)
    hipLaunchKernelGGL(maps_diff_norm_kernel, dim3((unsigned)(((long)T * H + 3) / 4)), dim3(256), 0, s, diff_out, diff_dtype, ldd, (const float*)out, ldo, lam, out_scale,
                       eps, T * H, H, DV);
  return launch_status();
}

int dihip_gqa_decode_step_supported(int H, int G, int D, int DV, int span_len, int cache_dtype, int rot_dims) {
  return cache_dtype == DIHIP_BF16 && G > 0 && H % G == 0 && H / G <= 16 && (D == 64 || D == 128) && (DV == 64 || DV == 128) && span_len % 64 == 0 && (rot_dims == 0 || rot_dims == D);
}

int dihip_gqa_decode_step(void* stream, void* out, int out_dtype, long ldo, const float* qkv, long ld, int q_off, int k_off, int v_off, const void* qnorm, const void* knorm,
                          int norm_dtype, float eps, const float* freq, int rot_dims, int layout, float mag, void* const* kspans, void* const* vspans, int span_stride,
                          int span_len, const void* sink, int w_dtype, int sink_mode, float softcap, const float* gate, long ldg, const int32_t* tok_pos,
                          const int32_t* ent_slot, const int32_t* ent_row0, int E, int T, int H, int G, int D, int DV, float scale, int nsplit, void* ws, size_t ws_bytes) {
  if (int rc = gqa_check("gqa_decode_step", out, out_dtype, ldo, qkv, ld, kspans, vspans, span_stride, span_len, sink, w_dtype, sink_mode, gate, ldg, H, G, D, DV, 1, 0)) return rc;
  DIHIP_REQUIRE(dihip_gqa_decode_step_supported(H, G, D, DV, span_len, DIHIP_BF16, rot_dims), DIHIP_PARAM_ERROR, "gqa_decode_step: %d heads over %d of %d / %d, rotation %d, span_len %d not served",
                H, G, D, DV, rot_dims, span_len);
  DIHIP_REQUIRE(E >= 0 && T >= E && tok_pos && ent_slot && ent_row0 && seq_dtype_ok(norm_dtype) && (rot_dims == 0 || freq) && (layout == 0 || layout == 1), DIHIP_PARAM_ERROR,
                "gqa_decode_step: bad argument");
  DIHIP_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && ld >= (long)q_off + (long)H * D && ld >= (long)k_off + (long)G * D && ld >= (long)v_off + (long)G * DV, DIHIP_PARAM_ERROR,
                "gqa_decode_step: columns outside the rows");
  DIHIP_REQUIRE(((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(qkv)) & 15u) == 0 && ldo % 4 == 0 && ld % 4 == 0 && q_off % 4 == 0, DIHIP_PARAM_ERROR,
                "gqa_decode_step: query and output rows in 16-byte pieces");
  DIHIP_REQUIRE(nsplit >= 1 && nsplit <= 1024 && (long)E * G <= INT32_MAX, DIHIP_PARAM_ERROR, "gqa_decode_step: bad split / request count");
  DIHIP_REQUIRE(ws_bytes >= dihip_gqa_attn_mc_workspace_bytes(T, H, DV, nsplit) && (nsplit == 1 || ws), DIHIP_PARAM_ERROR, "gqa_decode_step: workspace too small");
  if (E == 0) return DIHIP_SUCCESS;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  PrepArgs p{const_cast<float*>(qkv), ld, q_off, k_off, v_off, H, G, D, DV, G, qnorm, knorm, norm_dtype, eps, freq, rot_dims, layout, mag};
  GqaArgs a{out, out_dtype, ldo, nullptr, 0, kspans, vspans, span_stride, span_len, sink, w_dtype, sink_mode, softcap, gate, ldg, nullptr, tok_pos,
            ent_slot, ent_row0, nullptr, H, G, D, DV, scale, (float*)ws, T * H, 1, 0, 0};
  int rc = DIHIP_SUCCESS;
  auto go = [&](auto d, auto v) {
    constexpr int D_ = decltype(d)::value, V_ = decltype(v)::value;
    const size_t tiles = (size_t)4 * 64 * (D_ + V_) * 2, recs = (size_t)4 * 16 * (V_ + 4) * 4, bytes = tiles > recs ? tiles : recs;
    auto kern = softcap > 0.f ? gqa_decode_step_kernel<D_, V_, true> : gqa_decode_step_kernel<D_, V_, false>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
      rc = DIHIP_RUNTIME_ERROR;
      return;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(E * G), nsplit), dim3(256), bytes, s, p, a);
  };
  constexpr std::integral_constant<int, 64> c64{};
  constexpr std::integral_constant<int, 128> c128{};
  if (D == 64 && DV == 64) go(c64, c64);
  else if (D == 64) go(c64, c128);
  else if (DV == 64) go(c128, c64);
  else go(c128, c128);
  DIHIP_REQUIRE(rc == DIHIP_SUCCESS, DIHIP_RUNTIME_ERROR, "gqa_decode_step: LDS refused");
  if (nsplit > 1)
    hipLaunchKernelGGL(gqa_attn_merge_kernel, dim3(E * H), dim3(256), 0, s, out, out_dtype, ldo, (const float*)ws, nsplit, T * H, H, 1, DV, DV, gate, ldg, ent_row0);
  return launch_status();
}

int dihip_maps_diff_norm(void* stream, void* y, int y_dtype, long ldy, const float* x, long ldx, float lam, float out_scale, float eps, int T,
                         int H, int DV) {
  DIHIP_REQUIRE(T >= 0 && H > 0 && DV > 0 && y && x && ldy >= (long)H * DV && ldx >= (long)H * 2 * DV && seq_dtype_ok(y_dtype), DIHIP_PARAM_ERROR,
                "maps_diff_norm: bad argument");
  DIHIP_REQUIRE(DV <= 512, DIHIP_EXCEED_LIMIT_ERROR, "maps_diff_norm: heads of more than 512 values");
  if (T == 0) return DIHIP_SUCCESS;
  const long pairs = (long)T * H;
  hipLaunchKernelGGL(maps_diff_norm_kernel, dim3((unsigned)((pairs + 3) / 4)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), y, y_dtype, ldy,
                     x, ldx, lam, out_scale, eps, (int)pairs, H, DV);
  return launch_status();
}

}  // extern "C"
