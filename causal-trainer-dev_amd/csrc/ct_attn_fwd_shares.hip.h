// Attention forward for launches of few row blocks (32 query rows of one head).
//
// One workgroup of NW wavefronts per row block; wavefront w takes the pieces of 32 keys w, w + NW, ... and stages them in a
// region of LDS that is its own, so nothing in the loop waits for another wavefront: K's copies for the next piece go out as
// soon as the scores of this one are formed, V's behind the product with V. The sums are merged once, at the end, every
// wavefront adding its share of the columns. The time is that of the longest row's chain of pieces, each about
// 0.75 us at head dimension 64 and 0.95 at 128 for a lone wavefront (copies, 8 or 16 products, softmax, one after the other),
// and, where compute units hold all the workgroups that fit, of the 64 bytes a clock that reach a compute unit's LDS (8 or
// 16 KB per piece). What this replaces staged the keys of four wavefronts together, twice, with a barrier per step; at head
// dimension 128 a compute unit held one such workgroup, of these two. Measured, us (batch, row length, query / KV heads, head
// dimension; documents):
//   NW = 4: (2, 1024, 8/8, 128; 32-512) 13.9 -> 11.7      (1, 4096, 4/4, 128; 400-500) 14.2 -> 11.1
//           (4, 1024, 4/4, 128; rows)   16.5 -> 14.5      (1, 7168, 4/4, 64; rows)     68 -> 51
//           (2, 4480, 2/2, 64; images)  45 -> 30          (3, 2944, 24/8, 64)          42 / 57: not taken
//   NW = 8: (1, 2176, 2/2, 128; images) 23.4 -> 15.5      (1, 8192, 1/1, 128; rows)    83 -> 44
//           (1, 16384, 1/1, 64; rows)   106 -> 71
//   NW = 3: (1, 6144, 4/4, 128; rows)   91 -> 71          (1, 2048, 12/12, 128; 256-2048) 36.6 -> 28.7
//           (4, 1280, 4/4, 128; 400-500) 15.1 -> 12.3
// Two query blocks per wavefront, which would halve the copies, need more registers than there are (58 spilled, 1.5 to 2
// times as long); two short row blocks in one workgroup, found out from the bounds, wait for them first (9.5 -> 15.6 us).
#pragma once

#include "ct_attn_kernels.hip.h"

namespace ct {

// A wavefront's own piece of LDS: 32 keys' K rows, V rows and (twice, by turns) ids; in the end its share of the sums.
template <int D>
struct ShareRegion {
  static constexpr int kTileBytes = 32 * D * 2;
  static constexpr int kK = 0;
  static constexpr int kV = kTileBytes;
  static constexpr int kIds = 2 * kTileBytes;
  static constexpr int kSumBytes = 32 * D * 4;   // O^T, then m and l of the 64 lanes
  static constexpr int kBytes = kSumBytes + 512;
  static_assert(kIds + 256 <= kBytes, "the ids fit");
  static constexpr int kCopies = kTileBytes / 1024;  // per tile
};

// Copies 32 rows of D elements into the swizzled layout, by one wavefront.
template <int D>
struct WaveTileDma {
  static constexpr int CPR = D / 8, kRowsPerPass = 64 / CPR, kPasses = 32 / kRowsPerPass;
  unsigned lane_off[kPasses];
  CT_DEVICE explicit WaveTileDma(size_t row_stride_bytes) {
    const int l = lane_id();
#pragma unroll
    for (int n = 0; n < kPasses; ++n) {
      const int row = l / CPR + n * kRowsPerPass;
      lane_off[n] = (unsigned)(row * row_stride_bytes) + (unsigned)(((l % CPR) ^ swizzle<CPR>(row)) * 16);
    }
  }
  CT_DEVICE void issue(const char* origin, lds_addr tile) const {
#pragma unroll
    for (int n = 0; n < kPasses; ++n) dma16_s(origin, lane_off[n], tile + n * 1024);
  }
};

template <int N>
CT_DEVICE void wait_copies_but() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
CT_DEVICE void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int D, int NW>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2))) void
attn_fwd_shares_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  using Region = ShareRegion<D>;
  const lds_addr lds0 = lds_address_of(smem_raw);
  const int l = lane_id(), half = l >> 5, w = uniform(threadIdx.x >> 6);
  const lds_addr own = lds0 + w * Region::kBytes;
  // The head is the fast index, then the batch row, then the rank, longest row block first (as attn_fwd_split_kernel).
  const int nrb = p.S / 32, g = p.Hq / p.Hkv;
  const int group = blockIdx.x % p.Hq, pull = blockIdx.x / p.Hq;
  const int kvh = group % p.Hkv, h = kvh * g + group / p.Hkv;
  const int rank = pull / p.B, b = (pull + rank) % p.B;
  const int rb = uniform(meta_const(p.sched + query_schedule_offset(nrb, 1))[(size_t)b * schedule_ints(nrb) + rank]);

  RowBlockLoader<D> q_rows;
  q_rows.request(p.q + (((size_t)b * p.S + rb * 32) * p.Hq + h) * D, (size_t)p.Hq * D);
  const int pos = rb * 32 + (l & 31);
  const int* segb = p.seg + (size_t)b * p.S;
  const int seg_q = segb[pos];
  const int end_q = p.end ? p.end[(size_t)b * p.S + pos] : pos;
  const int* meta_b = p.meta + (size_t)b * nrb * kMetaW;
  const QueryBlockBounds mine = query_block_bounds(meta_b, rb);
  const bool any = mine.kv_first <= mine.kv_last;
  int t = any ? mine.kv_first * 2 + w : 0;           // pieces of 32 keys
  const int last = any ? mine.kv_last * 2 + 1 : -1;  // (S is a multiple of 128: every piece is whole)

  const size_t row_bytes = (size_t)p.Hkv * D * 2;
  const WaveTileDma<D> dma(row_bytes);
  const char* kbase = reinterpret_cast<const char*>(p.k + ((size_t)b * p.S * p.Hkv + kvh) * D);
  const char* vbase = reinterpret_cast<const char*>(p.v + ((size_t)b * p.S * p.Hkv + kvh) * D);
  auto issue_k = [&](int piece, int turn) {
    dma.issue(kbase + (size_t)piece * 32 * row_bytes, own + Region::kK);
    dma16_lanes_s(segb + piece * 32, (unsigned)l * 16, own + Region::kIds + turn * 128, 0xff);
  };
  auto issue_v = [&](int piece) { dma.issue(vbase + (size_t)piece * 32 * row_bytes, own + Region::kV); };
  auto piece_bounds = [&](int piece) {
    const MetaPtr m = meta_const(meta_b + piece * kMetaW);
    return KeyTileBounds{m[kMinNz], m[kMaxId], m[kUniform]};
  };

  KeyTileBounds ahead{};
  if (t <= last) {
    issue_k(t, 0);
    ahead = piece_bounds(t);
  }
  bf16x8 qf[D / 16];
  q_rows.to_fragments(own + Region::kV, qf);
  wait_lds_reads();
  if (t <= last) issue_v(t);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) qf[kk] = scale_bf16x8(qf[kk], p.scale);

  f32x16 oacc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db) oacc[db] = zero16();
  float m_run = kNegInf, l_run = 0.f;  // softmax reference (a recent running max, log2 domain), this lane's share of the sum
  const RowFragOffsets<D / 8> ro(own);
  const TrFragOffsets<D / 8, KSlots::kAccum> to(own);

  for (int turn = 0; t <= last; t += NW, turn ^= 1) {
    const bool more = t + NW <= last;
    const KeyTileBounds now = ahead;
    const int key0 = t * 32;
    if (!blocks_interact(mine.min_nz, mine.max_id, mine.end_max, uniform(now.min_nz), uniform(now.max_id), key0)) {
      wait_copies_but<0>();
      if (more) {
        ahead = piece_bounds(t + NW);
        issue_k(t + NW, turn ^ 1);
        issue_v(t + NW);
      }
      continue;
    }
    wait_copies_but<Region::kCopies>();  // K's and the ids'; behind them are V's
    f32x16 s = zero16();
    fragments_ahead<D / 16, 4>([&](int kk) { return ro.load(Region::kK, 0, kk); },
                               [&](int kk, bf16x8 k) { s = mfma32(k, qf[kk], s); });
    wait_lds_reads();
    if (more) issue_k(t + NW, turn ^ 1);
    // (a piece with one shared id turns the id test into a per-query predicate)
    const int k_uniform = uniform(now.uniform);
    if (mine.uniform == 0 || mine.uniform != k_uniform || key0 + 31 > mine.end_min) {
      const int seg_cmp = seg_q != 0 ? seg_q : -1;
      int last_rel = end_q - key0 - 4 * half;
      if (k_uniform == 0) {
        mask_block_t<true, true>(own + Region::kIds + turn * 128, seg_cmp, last_rel, 0, s);
      } else {
        if (seg_cmp != k_uniform) last_rel = -1;
        mask_block_t<false, true>(own, seg_cmp, last_rel, 0, s);
      }
    }
    // (Here, where no wait for LDS follows for a while: scalar loads count with LDS reads and return in any order.)
    if (more) ahead = piece_bounds(t + NW);
    float mx = kNegInf;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = pair_max(mx) * kLog2e;
    if (__any(mx > m_run + kRescaleSlack)) {  // (lazily, as attn_fwd_item)
      const float m_new = fmaxf(m_run, mx);
      const float alpha = exp2_fast(m_run - (m_new == kNegInf ? 0.f : m_new));
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
      m_run = m_new;
    }
    const float minus = m_run == kNegInf ? 0.f : -m_run;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = exp2_fast(fmaf(s[r], kLog2e, minus));
      psum += s[r];
    }
    l_run += psum;
    const bf16x8 pf[2] = {pack_acc8(s, 0), pack_acc8(s, 1)};
    if (more)
      wait_copies_but<Region::kCopies + 1>();  // V's; behind them are the next K's and ids'
    else
      wait_copies_but<0>();
    fragments_ahead<D / 16, 4>(
        [&](int i) { return to.load(Region::kV, i / (D / 32), i % (D / 32)); },
        [&](int i, bf16x8 v) { oacc[i % (D / 32)] = mfma32(v, pf[i / (D / 32)], oacc[i % (D / 32)]); });
    wait_lds_reads();
    if (more) issue_v(t + NW);
  }

  // Every share's sums go to its region (its copies have landed and been read), then each wavefront adds its part of
  // the columns over the shares, in a fixed order.
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd)
      lds_store<f32x4>(own + (db * 4 + qd) * 1024 + l * 16,
                       f32x4{oacc[db][4 * qd], oacc[db][4 * qd + 1], oacc[db][4 * qd + 2], oacc[db][4 * qd + 3]});
  lds_store<float>(own + Region::kSumBytes + l * 4, m_run);
  lds_store<float>(own + Region::kSumBytes + 256 + l * 4, l_run);
  __syncthreads();
  const lds_addr sums = lds0 + l * 16, stats = lds0 + Region::kSumBytes + l * 4;
  float by[NW], m_all = kNegInf, l_all = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    by[i] = lds_load<float>(stats + i * Region::kBytes);
    m_all = fmaxf(m_all, by[i]);
  }
  const float m_use = m_all == kNegInf ? 0.f : m_all;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    by[i] = exp2_fast(by[i] - m_use);
    l_all += by[i] * lds_load<float>(stats + i * Region::kBytes + 256);
  }
  const float l_tot = pair_sum(l_all);
  const bool has = l_tot > 0.f;
  const float inv = has ? 1.f / l_tot : 0.f;
  const size_t row = ((size_t)b * p.S + pos) * p.Hq + h;
  if (w == 0 && l < 32) p.lse[row] = has ? (__logf(l_tot) + m_all * kLn2) : 0.f;
  constexpr int kChunks = D / 8;  // of 8 columns
#pragma unroll
  for (int j = 0; j < (kChunks + NW - 1) / NW; ++j) {
    const int chunk = kChunks % NW == 0 ? w * (kChunks / NW) + j : w + j * NW;
    if (kChunks % NW != 0 && chunk >= kChunks) break;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const f32x4 x = lds_load<f32x4>(sums + i * Region::kBytes + chunk * 1024);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += x[e] * by[i];
    }
    *reinterpret_cast<bf16x4*>(p.out + row * D + chunk * 8 + 4 * half) =
        bf16x4{(bf16)(o[0] * inv), (bf16)(o[1] * inv), (bf16)(o[2] * inv), (bf16)(o[3] * inv)};
  }
}

}  // namespace ct
