// Attention forward, several workgroups per compute unit: head dimension 64, and head dimension 128
// where the launch is small or its rows are short.
//
// One workgroup of NW wavefronts per query tile, launched heaviest tile first and dealt by the
// hardware. Nothing runs in step across workgroups: what one of them spends on its prologue, its row
// maxima and its stores is another one's time on the matrix pipe, and no hand-written interleaving is
// needed. At head dimension 64 the loop is bound by the vector ALU (57 instructions, 16 of them exponentials, against 8 MFMAs
// per 32 keys of whole rows: 365 clocks for that mix by four wavefronts on end, 480 here; the matrix pipe is busy half of the
// time), and 4 wavefronts per SIMD at 104 registers keep it busy; the 8-wavefront workgroup in two half-step-shifted groups
// that this replaces had 2. The forms:
//
//   KS = 1  a wavefront takes all keys of its 32 query rows
//   KS = 2  two wavefronts share them, 32 keys each per step: half the chain of steps per row
//
// For KS = 2 the sums are merged through LDS at the end (in a fixed order). A step stages
// SUB x KS x KB x 32 keys; a wavefront works on KB x 32 of them at a time, SUB times. 32 at a time
// (KB = 1) keep the score registers few and skip what is masked in finer pieces.
//
// Measured, us (batch, row length, query / KV heads, head dimension, visible 64-key tiles per row on
// average): before = the 8-wavefront workgroups
//   (2, 4096, 8/8, 64, 4.2)        37.3 -> 20.4  KS = 2     (3, 2944, 24/8, 64, 5.7) 72.7 -> 45.4  KS = 2
//   (3, 4224, 48/8, 64, 2.3)      121.2 -> 68.9  KS = 1     (8, 4096, 32/8, 64, 32)   796 -> 660   KS = 1
//   (3, 2560, 8/8, 128, 7.8)       55.3 -> 42.0  KS = 2     (6, 1280, 32/16, 128, 0.4) 61.1 -> 46.2  KS = 1
// The maximum of a piece formed before its exponents / only where their sum asks for it, and padded row blocks through the loop / by
// themselves, us:
//   (8, 4096, 32/8, 64; rows) 608 / 590     (3, 2944, 24/8, 64; 40-2944) 39.5 / 38.7      (2, 1024, 8/8, 64; 32-512) 7.6 / 7.6
//   (3, 3072, 6/2, 128; images) 50.9 / 46.4 (4, 1024, 12/4, 128; 172-914) 21.4 / 20.5     (8, 640, 6/2, 64; 319-424) 9.0 / 9.1
#pragma once

#include "ct_attn_kernels.hip.h"

namespace ct {

template <int D, int NW, int KS, int KB, int SUB>
struct SplitStage {
  static_assert(KS <= 2, "the merge is one hand-over");
  static constexpr int kKeys = SUB * KS * KB * 32;  // keys per step
  static constexpr int kTileBytes = kKeys * D * 2;
  static constexpr int kK = 0;
  static constexpr int kV = kTileBytes;
  static constexpr int kSeg = 2 * kTileBytes;
  static constexpr int kBytes = 2 * kTileBytes + kKeys * 4;
  static constexpr int kTotalBytes = 2 * kBytes;
  static constexpr int kPatchBytes = 32 * D * 2;  // one wavefront's rows, on their way in and out
  static_assert(NW * kPatchBytes <= kBytes, "the Q rows pass through the second stage");
  // what a wavefront hands over: O^T and (m, l); half of the shares hand over at a time, in front of the store patches
  static constexpr int kMergeBytes = 64 * (D / 2 + 2) * 4;
  static constexpr int kStorePatches = NW / KS * (KS / 2) * kMergeBytes;
  static_assert(kStorePatches + NW / KS * kPatchBytes <= kTotalBytes, "the merge fits");
};

template <int D, int HS, int NW, int KS, int KB, int SUB>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : KB == 1 ? 3 : 2))) void
attn_fwd_split_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  const lds_addr lds0 = lds_address_of(smem_raw);
  using Stage = SplitStage<D, NW, KS, KB, SUB>;
  constexpr bool kSequences = D == 128 && KB == 2;  // the hand-scheduled MFMA sequences
  constexpr int kSlots = NW / KS, PB = kSlots / HS;  // row blocks of the workgroup, per head
  static_assert(PB * HS * KS == NW, "wavefronts = heads x row blocks x key shares");
  const int l = lane_id(), half = l >> 5, w = uniform(threadIdx.x >> 6);
  const int slot = w % kSlots, share = w / kSlots;
  const int nrb = p.S / 32, g = p.Hq / p.Hkv, slices = g / HS, groups = slices * p.Hkv;
  // The group is the fast index (a group stays on one XCD when they come in eights), then the batch
  // row, then the rank in the row's work-sorted schedule. The batch rows take turns in being first:
  // an XCD deals its workgroups to its four shader engines in turn, and with 4 rows in a fixed order
  // the row with the long documents would be one engine's alone (4 x 4096, 32/8 heads: 340 against 238 us).
  const int group = blockIdx.x % groups, pull = blockIdx.x / groups;
  const int kvh = group % p.Hkv, slice = group / p.Hkv;
  const int rank = pull / p.B, b = (pull + rank) % p.B;
  const int qt = uniform(meta_const(p.sched + query_schedule_offset(nrb, PB))[(size_t)b * schedule_ints(nrb) + rank]);
  const int h = kvh * g + slice * HS + slot % HS;
  const int rb = qt * PB + slot / HS;  // (S is a multiple of 128: every tile is whole)

  RowBlockLoader<D> q_rows;
  q_rows.request(p.q + (((size_t)b * p.S + rb * 32) * p.Hq + h) * D, (size_t)p.Hq * D);
  const int pos = rb * 32 + (l & 31);
  const int* segb = p.seg + (size_t)b * p.S;
  const int seg_q = segb[pos];
  const int end_q = p.end ? p.end[(size_t)b * p.S + pos] : pos;
  const int* meta_b = p.meta + (size_t)b * nrb * kMetaW;
  const QueryBlockBounds mine = query_block_bounds(meta_b, rb);
  int first_tile = INT_MAX, last_tile = -1;  // 64-key tiles, as the table has them
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const MetaPtr m = meta_const(meta_b + (qt * PB + i) * kMetaW);
    first_tile = min(first_tile, uniform(m[kKvFirst]));
    last_tile = max(last_tile, uniform(m[kKvLast]));
  }
  // (nor does a step of 64 or 128 keys leave the row)
  const bool any = first_tile <= last_tile;
  int t = any ? first_tile * 64 / Stage::kKeys : 0;
  const int last = any ? (last_tile * 64 + 63) / Stage::kKeys : -1;

  // Row blocks of padding (a quarter of the workgroups at (3, 2944, 24/8, 64), 6000 clocks each on the way below): zeros.
  if (!any) {
    if (share != 0) return;
    bf16* rows = p.out + (((size_t)b * p.S + rb * 32) * p.Hq + h) * D;
    constexpr int kPerRow = D / 8;
#pragma unroll
    for (int i = 0; i < 32 * kPerRow / 64; ++i)
      store_global16(rows + (size_t)(i * (64 / kPerRow) + l / kPerRow) * p.Hq * D + l % kPerRow * 8, u32x4{0, 0, 0, 0});
    if (l < 32) p.lse[((size_t)b * p.S + rb * 32 + l) * p.Hq + h] = 0.f;
    return;
  }
  const TileDma<Stage::kKeys, D / 8, NW * 64> dma((size_t)p.Hkv * D * 2);
  const char* kbase = reinterpret_cast<const char*>(p.k + ((size_t)b * p.S * p.Hkv + kvh) * D);
  const char* vbase = reinterpret_cast<const char*>(p.v + ((size_t)b * p.S * p.Hkv + kvh) * D);
  const size_t step_bytes = (size_t)p.Hkv * D * 2 * Stage::kKeys;
  auto issue = [&](int step, lds_addr stage) {
    dma.issue(kbase + (size_t)step * step_bytes, stage + Stage::kK);
    dma.issue(vbase + (size_t)step * step_bytes, stage + Stage::kV);
    if (threadIdx.x < Stage::kKeys / 4) dma16_s(segb + step * Stage::kKeys, threadIdx.x * 16, stage + Stage::kSeg);
  };
  // of the KB x 32 keys that this wavefront takes as its piece `sub` of a step
  auto piece_bounds = [&](int step, int sub) {
    const int piece = (step * KS + share) * SUB + sub;
    if constexpr (KB == 2) {
      return key_tile_bounds(meta_b, piece);
    } else {
      const MetaPtr m = meta_const(meta_b + piece * kMetaW);
      return KeyTileBounds{m[kMinNz], m[kMaxId], m[kUniform]};
    }
  };

  KeyTileBounds ahead[SUB];
  if (t <= last) {
    issue(t, lds0);
#pragma unroll
    for (int sub = 0; sub < SUB; ++sub) ahead[sub] = piece_bounds(t, sub);
  }
  bf16x8 qf[D / 16];
  q_rows.to_fragments(lds0 + (Stage::kBytes + w * Stage::kPatchBytes), qf);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) qf[kk] = scale_bf16x8(qf[kk], p.scale);

  f32x16 oacc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db) oacc[db] = zero16();
  // softmax reference (a recent running max, log2 domain) and the term of the exponents that it makes
  float m_run = kNegInf, minus_m = kUnseen;
  bool fresh = true;      // no piece yet
  float l_run = 0.f;      // this lane's share of the running sum
  const int own = share * SUB * KB * RowFragOffsets<D / 8>::kRowBlockBytes;  // this wavefront's keys in a stage
  RowFragOffsets<D / 8> ro(lds0 + own);
  TrFragOffsets<D / 8, KSlots::kAccum> to(lds0 + own);
  // (Opaque from here on: the compiler otherwise forms the fragments' addresses again in every step.)
  if constexpr (D == 64) {
#pragma unroll
    for (int k = 0; k < D / 16; ++k) asm volatile("" : "+v"(ro.ptr[k]));
#pragma unroll
    for (int second = 0; second < 2; ++second)
#pragma unroll
      for (int db = 0; db < D / 32; ++db) asm volatile("" : "+v"(to.ptr[second][db]));
  }

  // KB x 32 keys from `key0` on, at byte offset OFF of this wavefront's keys in LDS
  auto piece = [&](auto off_tag, const KeyTileBounds& keys, int key0, lds_addr ids) {
    constexpr int OFF = decltype(off_tag)::value;
    if (!blocks_interact(mine.min_nz, mine.max_id, mine.end_max, uniform(keys.min_nz), uniform(keys.max_id), key0)) return;
    f32x16 s[KB];
    if constexpr (kSequences) {
      qk_sequence_128<OFF + Stage::kK>(ro, qf, s);
    } else {
#pragma unroll
      for (int i = 0; i < KB; ++i) s[i] = zero16();
      if constexpr (KB == 1) {
        fragments_ahead<D / 16, 4>([&](int kk) { return ro.load(OFF + Stage::kK, 0, kk); },
                                   [&](int kk, bf16x8 k) { s[0] = mfma32(k, qf[kk], s[0]); });
      } else {
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
          for (int i = 0; i < KB; ++i) s[i] = mfma32(ro.load(OFF + Stage::kK, i, kk), qf[kk], s[i]);
      }
    }
    // (a piece with one shared id turns the id test into a per-query predicate)
    const int k_uniform = uniform(keys.uniform);
    const bool masked = mine.uniform == 0 || mine.uniform != k_uniform || key0 + KB * 32 - 1 > mine.end_min;
    if (masked) {
      const int seg_cmp = seg_q != 0 ? seg_q : -1;
      int last_rel = end_q - key0 - 4 * half;
      if (k_uniform == 0 && key0 + KB * 32 - 1 <= mine.end_min) {
#pragma unroll
        for (int i = 0; i < KB; ++i) mask_block_t<true, false>(ids, seg_cmp, last_rel, i, s[i]);
      } else if (k_uniform == 0) {
#pragma unroll
        for (int i = 0; i < KB; ++i) mask_block_t<true, true>(ids, seg_cmp, last_rel, i, s[i]);
      } else {
        if (seg_cmp != k_uniform) last_rel = -1;
#pragma unroll
        for (int i = 0; i < KB; ++i) mask_block_t<false, true>(ids, seg_cmp, last_rel, i, s[i]);
      }
    }
    f32x16 e[KB];
    auto exponents = [&] {
      float sum = -0.f;  // (the neutral element, so that the first addition falls away)
#pragma unroll
      for (int i = 0; i < KB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          e[i][r] = exp2_fast(fmaf(s[i][r], kLog2e, minus_m));
          sum += e[i][r];
        }
      return sum;
    };
    // Where the rows have a reference the sum of a piece says whether it has to move, and the maximum, 15 of 72 vector
    // instructions and a chain in front of the exponents, is formed only then; where rows are likely to see their first key (a
    // masked piece, or the first) it is formed at once. A sum that is infinite or no number asks for the maximum as well.
    float psum = 0.f;
    bool settled = !(masked || fresh);
    fresh = false;
    if (settled) {
      psum = exponents();
      settled = __builtin_amdgcn_ballot_w64(!(psum <= kMostSum)) == 0;
    }
    if (!settled) {
      float mx = kNegInf;
#pragma unroll
      for (int i = 0; i < KB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[i][r]);
      mx = pair_max(mx) * kLog2e;
      if (__any(mx > m_run + kMovesBy)) {
        const float m_new = fmaxf(m_run, mx);
        const float alpha = exp2_fast(m_run - (m_new == kNegInf ? 0.f : m_new));
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        m_run = m_new;
        minus_m = m_new == kNegInf ? kUnseen : -m_new;
      }
      psum = exponents();
    }
    l_run += psum;
    bf16x8 pf[2 * KB];
#pragma unroll
    for (int i = 0; i < 2 * KB; ++i) pf[i] = pack_acc8(e[i >> 1], i & 1);
    if constexpr (kSequences) {
      pv_sequence_128<OFF + Stage::kV>(to, pf, oacc);
    } else {
#pragma unroll
      for (int i = 0; i < 2 * KB; ++i)
#pragma unroll
        for (int db = 0; db < D / 32; ++db) oacc[db] = mfma32(to.load(OFF + Stage::kV, i, db), pf[i], oacc[db]);
    }
  };
  auto step = [&](auto stage_tag) {
    constexpr int CUR = decltype(stage_tag)::value;
    constexpr int kPieceBytes = KB * RowFragOffsets<D / 8>::kRowBlockBytes;
    // this step's copies have landed for every wavefront, and every wavefront has left the other stage
    dma_wait_all();
    __syncthreads();
    KeyTileBounds now[SUB];
#pragma unroll
    for (int sub = 0; sub < SUB; ++sub) now[sub] = ahead[sub];
    if (t < last) {
      issue(t + 1, lds0 + (CUR ^ 1) * Stage::kBytes);
#pragma unroll
      for (int sub = 0; sub < SUB; ++sub) ahead[sub] = piece_bounds(t + 1, sub);
    }
    const int first_key = (t * KS + share) * SUB * KB * 32;
    const lds_addr ids = lds0 + (CUR * Stage::kBytes + Stage::kSeg + share * SUB * KB * 128);
    piece(std::integral_constant<int, CUR * Stage::kBytes>{}, now[0], first_key, ids);
    if constexpr (SUB == 2)
      piece(std::integral_constant<int, CUR * Stage::kBytes + kPieceBytes>{}, now[1], first_key + KB * 32, ids + KB * 128);
    ++t;
  };
  while (t <= last) {
    step(std::integral_constant<int, 0>{});
    if (t > last) break;
    step(std::integral_constant<int, 1>{});
  }
  __syncthreads();  // the stages become hand-over space and store patches

  if constexpr (KS == 2) {  // share 1 of a row block hands its sums to share 0
    const lds_addr sums = lds0 + slot * Stage::kMergeBytes, row = sums + l * 16, stats = sums + D * 128 + l * 4;
    if (share == 1) {
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          lds_store<f32x4>(row + (db * 4 + qd) * 1024,
                           f32x4{oacc[db][4 * qd], oacc[db][4 * qd + 1], oacc[db][4 * qd + 2], oacc[db][4 * qd + 3]});
      lds_store<float>(stats, m_run);
      lds_store<float>(stats + 256, l_run);
    }
    __syncthreads();
    if (share != 0) return;
    const float m_other = lds_load<float>(stats), l_other = lds_load<float>(stats + 256);
    const float m_new = fmaxf(m_run, m_other);
    const float m_use = m_new == kNegInf ? 0.f : m_new;
    const float mine_by = exp2_fast(m_run - m_use), other_by = exp2_fast(m_other - m_use);
    l_run = l_run * mine_by + l_other * other_by;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const f32x4 o = lds_load<f32x4>(row + (db * 4 + qd) * 1024);
#pragma unroll
        for (int e = 0; e < 4; ++e) oacc[db][4 * qd + e] = oacc[db][4 * qd + e] * mine_by + o[e] * other_by;
      }
  }

  const float l_tot = pair_sum(l_run);
  const bool has = l_tot > 0.f;
  const float inv = has ? 1.f / l_tot : 0.f;
  if (l < 32) p.lse[((size_t)b * p.S + rb * 32 + l) * p.Hq + h] = has ? (__logf(l_tot) + m_run * kLn2) : 0.f;
  const lds_addr patch = lds0 + (Stage::kStorePatches + slot * Stage::kPatchBytes);
  store_rows_t<D>(oacc, inv, patch, p.out + (((size_t)b * p.S + rb * 32) * p.Hq + h) * D, (size_t)p.Hq * D);
}

}  // namespace ct
