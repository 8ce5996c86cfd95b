// The decoder-layer neighbours of the attention operator: reset position ids, the per-token
// rotary tables, partial rotary embedding of Q and K (both channel pairings, optionally fused
// with the bf16 pre-scale of Q that the attention operator otherwise does), and RMS
// normalisation forward and backward. All are single passes over HBM.
//
// Reference: src/modeling/rotary.py:82-110 (positions), :132-157 (tables), :113-129 and :160-204 (apply),
// src/modeling/architecture.py:155-162 (rms_norm).
#include "ct_error.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ct {

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ u32x4 as_u32x4(bf16x8 v) { return __builtin_bit_cast(u32x4, v); }

// One workgroup per batch row. A run starts at a valid position whose canonical id differs
// from its predecessor's or whose predecessor's id is 0 (position 0: predecessor id 0);
// position = index - index of the latest run start (running maximum), 0 where invalid.
__global__ __launch_bounds__(1024) void position_ids_kernel(const int* mask, const int* ids, int S,
                                                            int* out) {
  __shared__ int wave_max[16];
  __shared__ int carry_s;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nwaves = blockDim.x >> 6;
  const int* mrow = mask + (size_t)b * S;
  const int* irow = ids + (size_t)b * S;
  int* orow = out + (size_t)b * S;
  if (tid == 0) carry_s = 0;
  __syncthreads();
  for (int base = 0; base < S; base += blockDim.x) {
    const int s = base + tid;
    bool valid = false;
    int start_index = 0;
    if (s < S) {
      valid = mrow[s] != 0;
      const int prev = s > 0 ? irow[s - 1] : 0;
      if (valid && (irow[s] != prev || prev == 0)) start_index = s;
    }
    int incl = start_index;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int other = __shfl_up(incl, off, 64);
      if (lane >= off) incl = max(incl, other);
    }
    if (lane == 63) wave_max[wave] = incl;
    __syncthreads();
    int latest = carry_s;
    for (int k = 0; k < wave; ++k) latest = max(latest, wave_max[k]);
    latest = max(latest, incl);
    if (s < S) orow[s] = valid ? s - latest : 0;
    __syncthreads();
    if (tid == 0) {
      int total = carry_s;
      for (int k = 0; k < nwaves; ++k) total = max(total, wave_max[k]);
      carry_s = total;
    }
    __syncthreads();
  }
}

// cos / sin of f32(position) * inv_freq[p] evaluated in f32, rounded once to bf16.
__global__ __launch_bounds__(256) void rotary_tables_kernel(const int* positions,
                                                            const float* inv_freq, long tokens,
                                                            int pairs, bf16* cosine, bf16* sine) {
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= tokens * pairs) return;
  const long t = gid / pairs;
  const int p = (int)(gid % pairs);
  const float angle = (float)positions[t] * inv_freq[p];
  cosine[gid] = (bf16)cosf(angle);
  sine[gid] = (bf16)sinf(angle);
}

__device__ __forceinline__ bf16 scaled(bf16 v, float s, bool on) {
  return on ? (bf16)((float)v * s) : v;
}

// Rotary embedding in 16-byte chunks. A work item is one chunk (8 channels) of a head, Q heads first,
// then K heads, for TOKENS consecutive tokens. ADJACENT: pairs (2i, 2i+1), a chunk holds 4 pairs. Otherwise
// pairs (i, i + R/2): the item of a rotated chunk in the first half also handles the partner chunk, and
// the chunks of the second half are no items. Channels past the rotated ones are copied (and scaled).
// forward: out = bf16(bf16(R x) * s); inverse: out = bf16(R^T bf16(x * s)). The rotation is
// evaluated in f32 from the bf16 operands and rounded once.
//
// Bound by memory (each row read and written once, no 64-bit index arithmetic per chunk: a workgroup
// belongs to its tokens). With two tokens the rows of both are requested before the first is worked on,
// and head and chunk are found once for both; the size of a workgroup leaves no lane without an item
// where that is possible, and the second halves of rotated heads no longer idle. At 16384 tokens of 32 + 8
// heads of 128: adjacent pairs, 64 channels 65.5 -> 61.7 us (5.5 TB/s), halves 99.9 -> 74.5, halves of 128
// channels 85.6 -> 61.2 (one token: 62.6, 78.9, 60.2; four: 65.4, 76.7, 63.2).
constexpr int kRotaryTokens = 2;
template <bool ADJACENT, int TOKENS>
__global__ __launch_bounds__(512) void apply_rotary_kernel(ct_rotary_args a, int items_per_head, int items) {
  const int rot_chunks = a.rotary_pairs / 4;  // rotary_dim / 8
  const int half_chunks = rot_chunks / 2;
  const float s = (float)(bf16)a.q_scale;  // the scale is rounded to bf16 first
  const float sign = a.inverse ? -1.f : 1.f;
  const long t0 = (long)blockIdx.x * TOKENS;
  const int valid = a.tokens - t0 < TOKENS ? (int)(a.tokens - t0) : TOKENS;
  for (unsigned item = threadIdx.x; item < (unsigned)items; item += blockDim.x) {
    const int h = (int)(item / (unsigned)items_per_head);
    int c = (int)(item % (unsigned)items_per_head);
    if (!ADJACENT && c >= half_chunks) c += half_chunks;  // past the rotated channels
    const bool is_q = h < a.q_heads, rotated = c < rot_chunks;
    const size_t stride = (size_t)(is_q ? a.q_heads : a.kv_heads) * a.head_dim;  // of a token
    const size_t at = t0 * stride + (size_t)(is_q ? h : h - a.q_heads) * a.head_dim + c * 8;
    const uint16_t* in = (is_q ? a.q_in : a.k_in) + at;
    uint16_t* out = (is_q ? a.q_out : a.k_out) + at;
    const bool scale_on = is_q && a.q_scale != 1.0f;
    u32x4 x1[TOKENS], x2[TOKENS], cv[TOKENS], sv[TOKENS];
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
      const int t = min(k, valid - 1);
      x1[k] = *reinterpret_cast<const u32x4*>(in + t * stride);
      if (!rotated) continue;
      const uint16_t* cs = a.cosine + (t0 + t) * a.rotary_pairs;
      const uint16_t* sn = a.sine + (t0 + t) * a.rotary_pairs;
      if constexpr (ADJACENT) {
        const u32x2 c2 = *reinterpret_cast<const u32x2*>(cs + c * 4), s2 = *reinterpret_cast<const u32x2*>(sn + c * 4);
        cv[k] = u32x4{c2[0], c2[1], 0, 0};
        sv[k] = u32x4{s2[0], s2[1], 0, 0};
      } else {
        x2[k] = *reinterpret_cast<const u32x4*>(in + t * stride + half_chunks * 8);
        cv[k] = *reinterpret_cast<const u32x4*>(cs + c * 8);
        sv[k] = *reinterpret_cast<const u32x4*>(sn + c * 8);
      }
    }
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
      if (k >= valid) break;
      bf16x8 v = as_bf16x8(x1[k]), o;
      if (!rotated) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = scaled(v[e], s, scale_on);
      } else {
        const bf16x8 co8 = as_bf16x8(cv[k]), si8 = as_bf16x8(sv[k]);
        bf16x8 second = ADJACENT ? v : as_bf16x8(x2[k]), o2;
#pragma unroll
        for (int i = 0; i < (ADJACENT ? 4 : 8); ++i) {
          bf16 p = ADJACENT ? v[2 * i] : v[i], q = ADJACENT ? v[2 * i + 1] : second[i];
          if (a.inverse) {
            p = scaled(p, s, scale_on);
            q = scaled(q, s, scale_on);
          }
          const float co = (float)co8[i], si = sign * (float)si8[i];
          bf16 rp = (bf16)((float)p * co - (float)q * si);
          bf16 rq = (bf16)((float)q * co + (float)p * si);
          if (!a.inverse) {
            rp = scaled(rp, s, scale_on);
            rq = scaled(rq, s, scale_on);
          }
          if constexpr (ADJACENT) {
            o[2 * i] = rp;
            o[2 * i + 1] = rq;
          } else {
            o[i] = rp;
            o2[i] = rq;
          }
        }
        if constexpr (!ADJACENT) *reinterpret_cast<u32x4*>(out + k * stride + half_chunks * 8) = as_u32x4(o2);
      }
      *reinterpret_cast<u32x4*>(out + k * stride) = as_u32x4(o);
    }
  }
}

// Any head_dim and any even rotary dimension, one thread per (token, head) row and one channel
// pair at a time: the shapes the 16-byte kernel above does not take (e.g. 4 rotated channels of 8).
// Same arithmetic, element for element.
template <bool ADJACENT>
__global__ __launch_bounds__(256) void apply_rotary_rows_kernel(ct_rotary_args a) {
  const int heads = a.q_heads + a.kv_heads;
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= (long)a.tokens * heads) return;
  const long t = gid / heads;
  const int h = (int)(gid % heads);
  const bool is_q = h < a.q_heads;
  const bf16* in = reinterpret_cast<const bf16*>(is_q ? a.q_in : a.k_in);
  bf16* out = reinterpret_cast<bf16*>(is_q ? a.q_out : a.k_out);
  const size_t base = (is_q ? ((size_t)t * a.q_heads + h) : ((size_t)t * a.kv_heads + (h - a.q_heads))) * a.head_dim;
  const bool scale_on = is_q && a.q_scale != 1.0f;
  const float s = (float)(bf16)a.q_scale;
  const float sign = a.inverse ? -1.f : 1.f;
  const bf16* cs = reinterpret_cast<const bf16*>(a.cosine) + (size_t)t * a.rotary_pairs;
  const bf16* sn = reinterpret_cast<const bf16*>(a.sine) + (size_t)t * a.rotary_pairs;
  for (int i = 0; i < a.rotary_pairs; ++i) {
    const int c1 = ADJACENT ? 2 * i : i, c2 = ADJACENT ? 2 * i + 1 : i + a.rotary_pairs;
    bf16 x1 = in[base + c1], x2 = in[base + c2];
    if (a.inverse) {
      x1 = scaled(x1, s, scale_on);
      x2 = scaled(x2, s, scale_on);
    }
    const float co = (float)cs[i], si = sign * (float)sn[i];
    bf16 r1 = (bf16)((float)x1 * co - (float)x2 * si);
    bf16 r2 = (bf16)((float)x2 * co + (float)x1 * si);
    if (!a.inverse) {
      r1 = scaled(r1, s, scale_on);
      r2 = scaled(r2, s, scale_on);
    }
    out[base + c1] = r1;
    out[base + c2] = r2;
  }
  for (int c = 2 * a.rotary_pairs; c < a.head_dim; ++c) out[base + c] = scaled(in[base + c], s, scale_on);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// One wavefront per row: f32 mean of squares, r = 1 / sqrt(mean + eps),
// y = bf16(bf16(x r) * scale). The second pass over the row is served from cache.
__global__ __launch_bounds__(256) void rms_norm_fwd_kernel(const uint16_t* x, const uint16_t* scale,
                                                           float eps, long rows, int d, uint16_t* y,
                                                           float* rstd) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const uint16_t* xr = x + (size_t)row * d;
  float ss = 0.f;
  for (int c = lane; c < d / 8; c += 64) {
    const bf16x8 v = as_bf16x8(*reinterpret_cast<const u32x4*>(xr + c * 8));
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += (float)v[e] * (float)v[e];
  }
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)d + eps);
  if (rstd && lane == 0) rstd[row] = r;
  uint16_t* yr = y + (size_t)row * d;
  for (int c = lane; c < d / 8; c += 64) {
    const bf16x8 v = as_bf16x8(*reinterpret_cast<const u32x4*>(xr + c * 8));
    const bf16x8 w = as_bf16x8(*reinterpret_cast<const u32x4*>(scale + c * 8));
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (bf16)((float)(bf16)((float)v[e] * r) * (float)w[e]);
    *reinterpret_cast<u32x4*>(yr + c * 8) = as_u32x4(o);
  }
}

// The same for d <= 512 NCH with the row held in registers: every load of the row is in flight
// at once and x is read from memory exactly once.
template <int NCH>
__global__ __launch_bounds__(256) void rms_norm_fwd_rows_kernel(const uint16_t* x, const uint16_t* scale,
                                                                float eps, long rows, int d, uint16_t* y,
                                                                float* rstd) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63, chunks = d / 8;
  const uint16_t* xr = x + (size_t)row * d;
  u32x4 v[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    v[i] = i < NCH - 1 || lane + 64 * i < chunks ? *reinterpret_cast<const u32x4*>(xr + (lane + 64 * i) * 8) : u32x4{0, 0, 0, 0};
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += (float)as_bf16x8(v[i])[e] * (float)as_bf16x8(v[i])[e];
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)d + eps);
  if (rstd && lane == 0) rstd[row] = r;
  uint16_t* yr = y + (size_t)row * d;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    if (i == NCH - 1 && lane + 64 * i >= chunks) break;
    const bf16x8 w = as_bf16x8(*reinterpret_cast<const u32x4*>(scale + (lane + 64 * i) * 8));
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (bf16)((float)(bf16)((float)as_bf16x8(v[i])[e] * r) * (float)w[e]);
    *reinterpret_cast<u32x4*>(yr + (lane + 64 * i) * 8) = as_u32x4(o);
  }
}

// Backward of y = bf16(xhat) * w, xhat = x r: with g = dy w (f32),
//   dx = r (g - xhat mean(g xhat)) = r (g - xhat r mean(g x)),   dscale = sum over rows of dy bf16(xhat).
// WAVES wavefronts share a row (NCH chunks of 8 channels per lane, d <= 512 WAVES NCH), a workgroup takes
// 4 / WAVES rows at a time and keeps its share of dscale in registers; it leaves one f32 partial row that
// rms_norm_dscale_kernel adds up in workgroup order.
//
// Bound by memory: 6 bytes per element. With one wavefront per row and up to 320 registers the loads of a
// row waited for the two reductions of the row before (102 us at [16384, 4096]), and every wavefront
// left a partial row (32 MB written and read again). Sharing a row keeps a lane at 2 chunks, which leaves
// registers to load the next row ahead; both sums of a row travel in one reduction; hidden sizes
// that are not 512 times a power of two take the same kernel with the last chunk masked.
template <int WAVES, int NCH>
__global__ __launch_bounds__(256) void rms_norm_bwd_kernel(const uint16_t* x, const uint16_t* scale,
                                                           const uint16_t* dy, float eps, long rows, int d,
                                                           uint16_t* dx, float* partial) {
  constexpr int kRows = 4 / WAVES;  // rows a workgroup works on at a time
  __shared__ float exch[2][4][2];
  extern __shared__ float sums[];   // [kRows - 1][d] where several rows end in one partial row
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, part = wave % WAVES, chunks = d / 8;
  float acc[NCH][8];
  u32x4 w[NCH], xn[NCH], gn[NCH];
  int col[NCH];  // of chunk i, -1 past the row's end (only the last can be)
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[i][e] = 0.f;
    const int c = lane + 64 * (part + WAVES * i);
    col[i] = c < chunks ? c * 8 : -1;
    w[i] = col[i] >= 0 ? *reinterpret_cast<const u32x4*>(scale + col[i]) : u32x4{0, 0, 0, 0};
  }
  auto fetch = [&](long row) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const bool in = row < rows && col[i] >= 0;
      xn[i] = in ? *reinterpret_cast<const u32x4*>(x + (size_t)row * d + col[i]) : u32x4{0, 0, 0, 0};
      gn[i] = in ? *reinterpret_cast<const u32x4*>(dy + (size_t)row * d + col[i]) : u32x4{0, 0, 0, 0};
    }
  };
  const long stride = (long)gridDim.x * kRows;
  long row = (long)blockIdx.x * kRows + wave / WAVES;
  fetch(row);
  // (all wavefronts of a workgroup take the same number of turns: the barrier below is uniform)
  for (long base = (long)blockIdx.x * kRows, turn = 0; base < rows; base += stride, row += stride, ++turn) {
    u32x4 xv[NCH], gv[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      xv[i] = xn[i];
      gv[i] = gn[i];
    }
    fetch(row + stride);
    float ss = 0.f, dot = 0.f;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xf = (float)as_bf16x8(xv[i])[e];
        ss += xf * xf;
        dot += (float)as_bf16x8(gv[i])[e] * (float)as_bf16x8(w[i])[e] * xf;
      }
    ss = wave_sum(ss);
    dot = wave_sum(dot);
    if constexpr (WAVES > 1) {
      float (*e)[2] = exch[turn & 1];  // (two of them: one barrier per turn)
      if (lane == 0) {
        e[wave][0] = ss;
        e[wave][1] = dot;
      }
      __syncthreads();
      ss = dot = 0.f;
#pragma unroll
      for (int k = 0; k < WAVES; ++k) {
        ss += e[wave / WAVES * WAVES + k][0];
        dot += e[wave / WAVES * WAVES + k][1];
      }
    }
    const float r = 1.0f / sqrtf(ss / (float)d + eps);
    const float mean = dot * r / (float)d;
    if (row < rows) {
      uint16_t* dr = dx + (size_t)row * d;
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        if (col[i] < 0) continue;
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float xhat = (float)as_bf16x8(xv[i])[e] * r, g = (float)as_bf16x8(gv[i])[e];
          acc[i][e] += g * (float)(bf16)xhat;
          o[e] = (bf16)(r * (g * (float)as_bf16x8(w[i])[e] - xhat * mean));
        }
        *reinterpret_cast<u32x4*>(dr + col[i]) = as_u32x4(o);
      }
    }
  }
  // the workgroup's row groups, in order
  float* prow = partial + (size_t)blockIdx.x * d;
  if constexpr (kRows > 1) {
    if (wave >= WAVES) {
      float* mine = sums + (size_t)(wave / WAVES - 1) * d;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
        if (col[i] >= 0)
#pragma unroll
          for (int e = 0; e < 8; ++e) mine[col[i] + e] = acc[i][e];
    }
    __syncthreads();
    if (wave >= WAVES) return;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (col[i] >= 0)
#pragma unroll
        for (int k = 0; k < kRows - 1; ++k)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[i][e] += sums[(size_t)k * d + col[i] + e];
  }
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (col[i] >= 0) {
      *reinterpret_cast<f32x4*>(prow + col[i]) = f32x4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
      *reinterpret_cast<f32x4*>(prow + col[i] + 4) = f32x4{acc[i][4], acc[i][5], acc[i][6], acc[i][7]};
    }
}

// The same with the forward's r of every row, for few of them: dx and dscale then have nothing to wait for in each other and
// are one launch. Workgroups before column_groups add 32 columns of dscale over all rows (8 columns of every 64th row a
// thread, the 16 rows of a wavefront, the wavefronts, in that order), the others form dx of 4 / WAVES rows.
// Bound by latency: us of the two kernels above and below without the wait between them / of this one, [260, 1024] 6.2 / 4.8,
// [4, 512] 4.2 / 3.6, [1024, 512] 6.1 / 6.8, [512, 4096] 10.8 / 6.6, [1024, 8192] 21.7 / 18.4; the launch saved is 2 us of a
// host that does not keep ahead (norm and rotary on [2, 130, 1024], both directions, 90.6 / 88.8; on [4, 128, 4096] 90.8 / 88.4). More rows lose: [2048, 512]
// 7.6 / 10.0, [2048, 2048] 13.3 / 17.8, [4096, 1024] 12.0 / 29.4. (Every column group forming r by itself: [260, 1024] 14.9.)
template <int WAVES, int NCH>
__global__ __launch_bounds__(256) void rms_norm_bwd_saved_kernel(const uint16_t* x, const uint16_t* scale, const uint16_t* dy,
                                                                 const float* rstd, int rows, int d, int column_groups, uint16_t* dx,
                                                                 bf16* dscale) {
  __shared__ float exch[4][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if ((int)blockIdx.x < column_groups) {
    const int col = (int)blockIdx.x * 32 + (threadIdx.x & 3) * 8;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    if (col < d) {
#pragma unroll 4
      for (int row = threadIdx.x >> 2; row < rows; row += 64) {
        const bf16x8 xv = as_bf16x8(*reinterpret_cast<const u32x4*>(x + (size_t)row * d + col));
        const bf16x8 gv = as_bf16x8(*reinterpret_cast<const u32x4*>(dy + (size_t)row * d + col));
        const float r = rstd[row];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += (float)gv[e] * (float)(bf16)((float)xv[e] * r);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int off = 32; off >= 4; off >>= 1) acc[e] += __shfl_xor(acc[e], off, 64);
      if (lane < 4) exch[wave][lane * 8 + e] = acc[e];
    }
    __syncthreads();
    const int out = (int)blockIdx.x * 32 + threadIdx.x;
    if (threadIdx.x < 32 && out < d)
      dscale[out] = (bf16)((exch[0][threadIdx.x] + exch[1][threadIdx.x]) + (exch[2][threadIdx.x] + exch[3][threadIdx.x]));
    return;
  }
  const int part = wave % WAVES, chunks = d / 8, row = ((int)blockIdx.x - column_groups) * (4 / WAVES) + wave / WAVES;
  u32x4 w[NCH], xv[NCH], gv[NCH];
  float dot = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = lane + 64 * (part + WAVES * i);
    const bool in = row < rows && c < chunks;
    w[i] = in ? *reinterpret_cast<const u32x4*>(scale + c * 8) : u32x4{0, 0, 0, 0};
    xv[i] = in ? *reinterpret_cast<const u32x4*>(x + (size_t)row * d + c * 8) : u32x4{0, 0, 0, 0};
    gv[i] = in ? *reinterpret_cast<const u32x4*>(dy + (size_t)row * d + c * 8) : u32x4{0, 0, 0, 0};
  }
  const float r = row < rows ? rstd[row] : 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) dot += (float)as_bf16x8(gv[i])[e] * (float)as_bf16x8(w[i])[e] * (float)as_bf16x8(xv[i])[e];
  dot = wave_sum(dot);
  if constexpr (WAVES > 1) {
    if (lane == 0) exch[wave][0] = dot;
    __syncthreads();
    dot = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) dot += exch[wave / WAVES * WAVES + k][0];
  }
  const float mean = dot * r / (float)d;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = lane + 64 * (part + WAVES * i);
    if (row >= rows || c >= chunks) continue;
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      o[e] = (bf16)(r * ((float)as_bf16x8(gv[i])[e] * (float)as_bf16x8(w[i])[e] - (float)as_bf16x8(xv[i])[e] * r * mean));
    *reinterpret_cast<u32x4*>(dx + (size_t)row * d + c * 8) = as_u32x4(o);
  }
}

// Hidden sizes past 8192: the row is walked three times (sum of squares, the
// dot product, dx; the repeats are served from cache) and the wavefront's dscale sums live in its
// row of `partial` instead of registers (a lane only ever touches its own columns of it).
__global__ __launch_bounds__(256) void rms_norm_bwd_any_kernel(const uint16_t* x, const uint16_t* scale,
                                                               const uint16_t* dy, float eps, long rows, int d,
                                                               uint16_t* dx, float* partial) {
  const int lane = threadIdx.x & 63, chunks = d / 8;
  const long wv = (long)blockIdx.x * 4 + (threadIdx.x >> 6), waves = (long)gridDim.x * 4;
  float* prow = partial + (size_t)wv * d;
  for (int c = lane; c < chunks; c += 64)
#pragma unroll
    for (int e = 0; e < 8; ++e) prow[c * 8 + e] = 0.f;
  for (long row = wv; row < rows; row += waves) {
    const uint16_t* xr = x + (size_t)row * d;
    const uint16_t* gr = dy + (size_t)row * d;
    float ss = 0.f;
    for (int c = lane; c < chunks; c += 64) {
      const bf16x8 xv = as_bf16x8(*reinterpret_cast<const u32x4*>(xr + c * 8));
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += (float)xv[e] * (float)xv[e];
    }
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / (float)d + eps);
    float dot = 0.f;
    for (int c = lane; c < chunks; c += 64) {
      const bf16x8 xv = as_bf16x8(*reinterpret_cast<const u32x4*>(xr + c * 8));
      const bf16x8 gv = as_bf16x8(*reinterpret_cast<const u32x4*>(gr + c * 8));
      const bf16x8 wv8 = as_bf16x8(*reinterpret_cast<const u32x4*>(scale + c * 8));
#pragma unroll
      for (int e = 0; e < 8; ++e) dot += (float)gv[e] * (float)wv8[e] * ((float)xv[e] * r);
    }
    dot = wave_sum(dot) / (float)d;
    uint16_t* dr = dx + (size_t)row * d;
    for (int c = lane; c < chunks; c += 64) {
      const bf16x8 xv = as_bf16x8(*reinterpret_cast<const u32x4*>(xr + c * 8));
      const bf16x8 gv = as_bf16x8(*reinterpret_cast<const u32x4*>(gr + c * 8));
      const bf16x8 wv8 = as_bf16x8(*reinterpret_cast<const u32x4*>(scale + c * 8));
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xhat = (float)xv[e] * r;
        o[e] = (bf16)(r * ((float)gv[e] * (float)wv8[e] - xhat * dot));
        prow[c * 8 + e] += (float)gv[e] * (float)(bf16)xhat;
      }
      *reinterpret_cast<u32x4*>(dr + c * 8) = as_u32x4(o);
    }
  }
}

// dscale[col] = sum of the partial rows in a fixed order: thread (c, g) adds the rows g, g + 32, ... for
// column 32 blockIdx.x + c (four independent chains, joined in order), then the 32 group sums are added
// in order. Exactly one of the two outputs is given.
__global__ __launch_bounds__(1024) void rms_norm_dscale_kernel(const float* partial, int count, int d,
                                                               float* dscale, bf16* dscale_rounded) {
  __shared__ float group[32][33];
  const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int col = blockIdx.x * 32 + c;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (col < d) {
    const float* p = partial + col;
    int i = g;
    for (; i + 96 < count; i += 128) {
      s0 += p[(size_t)i * d];
      s1 += p[(size_t)(i + 32) * d];
      s2 += p[(size_t)(i + 64) * d];
      s3 += p[(size_t)(i + 96) * d];
    }
    for (; i < count; i += 32) s0 += p[(size_t)i * d];
  }
  group[g][c] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (g == 0 && col < d) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 32; ++k) s += group[k][c];
    if (dscale) dscale[col] = s;
    else dscale_rounded[col] = (bf16)s;
  }
}

// Partial rows of dscale: three workgroups per compute unit, as many as the registers of a shared row
// leave room for (the walking kernel writes one per wavefront).
constexpr int kNormBwdBlocks = 768;
constexpr int kNormBwdAnyBlocks = 512;
// The line: the threads of a column group walk rows / 64 rows each, and x and dy are read twice (figures at the kernel).
constexpr long kNormSavedRows = 1024;

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace ct

using namespace ct;

extern "C" int32_t ct_position_ids(void* stream, const int32_t* attention_mask,
                                   const int32_t* canonical_ids, int32_t batch, int32_t seq,
                                   int32_t* position_ids) {
  CT_REQUIRE(attention_mask && canonical_ids && position_ids, "ct_position_ids: null pointer");
  CT_REQUIRE(batch > 0 && seq > 0, "ct_position_ids: batch and sequence must be positive, got [%d, %d]",
             batch, seq);
  const int threads = seq >= 1024 ? 1024 : ((seq + 63) / 64) * 64;
  LaunchScope scope("position_ids_kernel", (hipStream_t)stream);
  hipLaunchKernelGGL(position_ids_kernel, dim3(batch), dim3(threads), 0, (hipStream_t)stream,
                     attention_mask, canonical_ids, seq, position_ids);
  return scope.done();
}

extern "C" int32_t ct_rotary_cos_sin(void* stream, const int32_t* position_ids, const float* inv_freq,
                                     int64_t tokens, int32_t rotary_pairs, uint16_t* cosine,
                                     uint16_t* sine) {
  CT_REQUIRE(position_ids && inv_freq && cosine && sine, "ct_rotary_cos_sin: null pointer");
  CT_REQUIRE(tokens > 0, "ct_rotary_cos_sin: token count must be positive");
  CT_REQUIRE(rotary_pairs > 0, "ct_rotary_cos_sin: inv_freq must be a non-empty vector");
  const long total = (long)tokens * rotary_pairs;
  LaunchScope scope("rotary_tables_kernel", (hipStream_t)stream);
  hipLaunchKernelGGL(rotary_tables_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, position_ids, inv_freq, (long)tokens, rotary_pairs,
                     reinterpret_cast<bf16*>(cosine), reinterpret_cast<bf16*>(sine));
  return scope.done();
}

extern "C" int32_t ct_apply_rotary(void* stream, const ct_rotary_args* a) {
  CT_REQUIRE(a, "ct_apply_rotary: null args");
  CT_REQUIRE(a->q_in && a->k_in && a->q_out && a->k_out && a->cosine && a->sine,
             "ct_apply_rotary: null pointer");
  CT_REQUIRE(a->tokens > 0 && a->q_heads > 0 && a->kv_heads > 0 && a->head_dim > 0,
             "ct_apply_rotary: dimensions must be positive");
  CT_REQUIRE(a->rope_style == CT_ROPE_GPT_J || a->rope_style == CT_ROPE_GPT_NEOX,
             "ct_apply_rotary: rope_style must be 'gpt-j' or 'gpt-neox'");
  const int rotary_dim = 2 * a->rotary_pairs;
  CT_REQUIRE(a->rotary_pairs > 0 && rotary_dim <= a->head_dim,
             "ct_apply_rotary: invalid rotary dimension %d for head_dim=%d", rotary_dim, a->head_dim);
  const bool vector_path = a->head_dim % 8 == 0 && rotary_dim % 16 == 0;
  CT_REQUIRE(a->q_scale == a->q_scale && a->q_scale - a->q_scale == 0.f,
             "ct_apply_rotary: q_scale must be finite");
  CT_REQUIRE(!vector_path || (aligned16(a->q_in) && aligned16(a->k_in) && aligned16(a->q_out) && aligned16(a->k_out) &&
                              aligned16(a->cosine) && aligned16(a->sine)),
             "ct_apply_rotary: pointers must be 16-byte aligned");
  CT_REQUIRE(a->tokens <= 0x7fffffffll, "ct_apply_rotary: at most 2^31 - 1 tokens per call");
  LaunchScope scope("apply_rotary_kernel", (hipStream_t)stream);
  if (!vector_path) {
    // head_dim not a multiple of 8 or fewer than 16 rotated channels at a time: element-wise kernel
    const long rows = (long)a->tokens * (a->q_heads + a->kv_heads);
    const dim3 grid((unsigned)((rows + 255) / 256));
    if (a->rope_style == CT_ROPE_GPT_J)
      hipLaunchKernelGGL((apply_rotary_rows_kernel<true>), grid, dim3(256), 0, (hipStream_t)stream, *a);
    else
      hipLaunchKernelGGL((apply_rotary_rows_kernel<false>), grid, dim3(256), 0, (hipStream_t)stream, *a);
    return scope.done();
  }
  const bool adjacent = a->rope_style == CT_ROPE_GPT_J;
  const int per_head = a->head_dim / 8 - (adjacent ? 0 : a->rotary_pairs / 8), items = (a->q_heads + a->kv_heads) * per_head;
  // as many threads as leave the fewest idle in the last round (640 items: 320), the most of those
  int threads = 64;
  for (int n = 128; n <= 512; n += 64)
    if ((items + n - 1) / n * n <= (items + threads - 1) / threads * threads) threads = n;
  // several tokens a workgroup once every compute unit has 8 workgroups of them
  const int tokens = a->tokens >= 256 * 8 * kRotaryTokens ? kRotaryTokens : 1;
  const dim3 grid((unsigned)((a->tokens + tokens - 1) / tokens)), block(threads);
  hipStream_t st = (hipStream_t)stream;
  if (adjacent && tokens == 1) hipLaunchKernelGGL((apply_rotary_kernel<true, 1>), grid, block, 0, st, *a, per_head, items);
  else if (adjacent) hipLaunchKernelGGL((apply_rotary_kernel<true, kRotaryTokens>), grid, block, 0, st, *a, per_head, items);
  else if (tokens == 1) hipLaunchKernelGGL((apply_rotary_kernel<false, 1>), grid, block, 0, st, *a, per_head, items);
  else hipLaunchKernelGGL((apply_rotary_kernel<false, kRotaryTokens>), grid, block, 0, st, *a, per_head, items);
  return scope.done();
}

extern "C" int32_t ct_rms_norm_fwd(void* stream, const uint16_t* x, const uint16_t* scale, float eps,
                                   int64_t rows, int32_t hidden, uint16_t* y, float* rstd) {
  CT_REQUIRE(x && scale && y, "ct_rms_norm_fwd: null pointer");
  CT_REQUIRE(rows > 0 && hidden > 0 && hidden % 8 == 0,
             "ct_rms_norm_fwd: rows must be positive and the hidden size a multiple of 8, got [%lld, %d]",
             (long long)rows, hidden);
  CT_REQUIRE(aligned16(x) && aligned16(scale) && aligned16(y),
             "ct_rms_norm_fwd: pointers must be 16-byte aligned");
  LaunchScope scope("rms_norm_fwd_kernel", (hipStream_t)stream);
  const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
  hipStream_t st = (hipStream_t)stream;
  const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, x, scale, eps, (long)rows, hidden, y, rstd); };
  // Rows in registers up to 4096 channels and around the two larger sizes that models have, 5120 and 8192 (an instance
  // per 512 channels); rows of 4104 to 4608, 5128 to 7680 and more than 8192 are walked twice, the second
  // time from cache.
  switch (int chunks = (hidden + 511) / 512; chunks) {
    case 1: launch(rms_norm_fwd_rows_kernel<1>); break;
    case 2: launch(rms_norm_fwd_rows_kernel<2>); break;
    case 3: launch(rms_norm_fwd_rows_kernel<3>); break;
    case 4: launch(rms_norm_fwd_rows_kernel<4>); break;
    case 5: launch(rms_norm_fwd_rows_kernel<5>); break;
    case 6: launch(rms_norm_fwd_rows_kernel<6>); break;
    case 7: launch(rms_norm_fwd_rows_kernel<7>); break;
    case 8: launch(rms_norm_fwd_rows_kernel<8>); break;
    case 10: launch(rms_norm_fwd_rows_kernel<10>); break;
    case 16: launch(rms_norm_fwd_rows_kernel<16>); break;
    default: launch(rms_norm_fwd_kernel);
  }
  return scope.done();
}

extern "C" size_t ct_rms_norm_bwd_workspace_bytes(int32_t hidden) {
  if (hidden <= 0) return 0;
  return (size_t)(hidden <= 8192 ? kNormBwdBlocks : kNormBwdAnyBlocks * 4) * hidden * sizeof(float);
}

// Wavefronts that share a row of up to 8192: the fewest that keep a lane at 2 chunks (3 or 4 past 4096).
static int norm_bwd_waves(int hidden) { return hidden <= 1024 ? 1 : hidden <= 2048 ? 2 : 4; }

static int32_t rms_norm_bwd_on(void* stream_, const uint16_t* x, const uint16_t* scale, const uint16_t* dy, float eps,
                               int64_t rows, int32_t hidden, uint16_t* dx, float* dscale, uint16_t* dscale_rounded,
                               void* workspace, size_t workspace_bytes) {
  CT_REQUIRE(x && scale && dy && dx && (dscale || dscale_rounded) && workspace, "ct_rms_norm_bwd: null pointer");
  CT_REQUIRE(rows > 0, "ct_rms_norm_bwd: rows must be positive");
  CT_REQUIRE(hidden > 0 && hidden % 8 == 0, "ct_rms_norm_bwd: hidden size must be a multiple of 8, got %d", hidden);
  CT_REQUIRE(aligned16(x) && aligned16(scale) && aligned16(dy) && aligned16(dx) && aligned16(workspace),
             "ct_rms_norm_bwd: pointers must be 16-byte aligned");
  if (workspace_bytes < ct_rms_norm_bwd_workspace_bytes(hidden))
    return fail(CT_WORKSPACE_TOO_SMALL, "ct_rms_norm_bwd: workspace %zu < %zu bytes", workspace_bytes,
                ct_rms_norm_bwd_workspace_bytes(hidden));
  hipStream_t stream = (hipStream_t)stream_;
  float* partial = static_cast<float*>(workspace);
  int count;  // partial rows
  LaunchScope scope("rms_norm_bwd_kernel", stream);
  if (hidden > 8192) {
    hipLaunchKernelGGL(rms_norm_bwd_any_kernel, dim3(kNormBwdAnyBlocks), dim3(256), 0, stream, x, scale, dy, eps, (long)rows,
                       hidden, dx, partial);
    count = kNormBwdAnyBlocks * 4;
  } else {
    const int waves = norm_bwd_waves(hidden), at_a_time = 4 / waves;
    const int64_t groups = (rows + at_a_time - 1) / at_a_time;
    count = groups < kNormBwdBlocks ? (int)groups : kNormBwdBlocks;
    const size_t smem = (size_t)(at_a_time - 1) * hidden * sizeof(float);
    const auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(count), dim3(256), smem, stream, x, scale, dy, eps, (long)rows, hidden, dx, partial);
    };
    switch (int chunks = (hidden + 512 * waves - 1) / (512 * waves); 8 * waves + chunks) {
      case 9: launch(rms_norm_bwd_kernel<1, 1>); break;
      case 10: launch(rms_norm_bwd_kernel<1, 2>); break;
      case 18: launch(rms_norm_bwd_kernel<2, 2>); break;
      case 34: launch(rms_norm_bwd_kernel<4, 2>); break;
      case 35: launch(rms_norm_bwd_kernel<4, 3>); break;
      default: launch(rms_norm_bwd_kernel<4, 4>); break;
    }
  }
  int rc = scope.done();
  if (rc) return rc;
  LaunchScope scope2("rms_norm_dscale_kernel", stream);
  hipLaunchKernelGGL(rms_norm_dscale_kernel, dim3((hidden + 31) / 32), dim3(1024), 0, stream, partial, count, hidden, dscale,
                     reinterpret_cast<bf16*>(dscale_rounded));
  return scope2.done();
}

extern "C" int32_t ct_rms_norm_keeps_rstd(int64_t rows, int32_t hidden) {
  return rows > 0 && rows <= kNormSavedRows && hidden > 0 && hidden <= 8192 && hidden % 8 == 0;
}

extern "C" int32_t ct_rms_norm_bwd_saved(void* stream_, const uint16_t* x, const uint16_t* scale, const uint16_t* dy,
                                         const float* rstd, int64_t rows, int32_t hidden, uint16_t* dx, uint16_t* dscale) {
  CT_REQUIRE(x && scale && dy && rstd && dx && dscale, "ct_rms_norm_bwd_saved: null pointer");
  CT_REQUIRE(ct_rms_norm_keeps_rstd(rows, hidden), "ct_rms_norm_bwd_saved: not a size that keeps rstd, got [%lld, %d]",
             (long long)rows, hidden);
  CT_REQUIRE(aligned16(x) && aligned16(scale) && aligned16(dy) && aligned16(dx), "ct_rms_norm_bwd_saved: pointers must be 16-byte aligned");
  hipStream_t stream = (hipStream_t)stream_;
  LaunchScope scope("rms_norm_bwd_saved_kernel", stream);
  const int waves = norm_bwd_waves(hidden), column_groups = (hidden + 31) / 32;
  const int row_groups = ((int)rows + 4 / waves - 1) / (4 / waves);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(column_groups + row_groups), dim3(256), 0, stream, x, scale, dy, rstd, (int)rows, hidden,
                       column_groups, dx, reinterpret_cast<bf16*>(dscale));
  };
  switch (int chunks = (hidden + 512 * waves - 1) / (512 * waves); 8 * waves + chunks) {
    case 9: launch(rms_norm_bwd_saved_kernel<1, 1>); break;
    case 10: launch(rms_norm_bwd_saved_kernel<1, 2>); break;
    case 18: launch(rms_norm_bwd_saved_kernel<2, 2>); break;
    case 34: launch(rms_norm_bwd_saved_kernel<4, 2>); break;
    case 35: launch(rms_norm_bwd_saved_kernel<4, 3>); break;
    default: launch(rms_norm_bwd_saved_kernel<4, 4>); break;
  }
  return scope.done();
}

extern "C" int32_t ct_rms_norm_bwd(void* stream, const uint16_t* x, const uint16_t* scale, const uint16_t* dy, float eps,
                                   int64_t rows, int32_t hidden, uint16_t* dx, float* dscale, void* workspace,
                                   size_t workspace_bytes) {
  return rms_norm_bwd_on(stream, x, scale, dy, eps, rows, hidden, dx, dscale, nullptr, workspace, workspace_bytes);
}

extern "C" int32_t ct_rms_norm_bwd_rounded(void* stream, const uint16_t* x, const uint16_t* scale, const uint16_t* dy,
                                           float eps, int64_t rows, int32_t hidden, uint16_t* dx, uint16_t* dscale,
                                           void* workspace, size_t workspace_bytes) {
  return rms_norm_bwd_on(stream, x, scale, dy, eps, rows, hidden, dx, nullptr, dscale, workspace, workspace_bytes);
}
