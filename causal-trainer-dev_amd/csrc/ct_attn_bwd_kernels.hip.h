// Attention backward kernels for gfx950.
//
// dQ kernel: same walk as the forward (a wavefront owns 32 query rows and
// visits the 64-key tiles they can see). Per tile, transposed:
//   S^T = K Q^T, P^T = exp(S^T - lse), dP^T = V dO^T, dS^T = P^T (dP^T - delta),
//   dQ^T += K^T dS^T                      (src/kernels/efficient_attention.py:1015-1048)
// dK/dV kernel: a workgroup owns 128 keys of one KV head (32 per wavefront,
// K and V fragments held in registers) and walks every (query head of the
// group, 32-row query block) that can see them; Q (pre-scaled, bf16) and dO
// are staged through LDS. Per block:
//   S = Q K^T, P = exp(S - lse), dP = dO V^T, dS = P (dP - delta),
//   dV += P^T dO, dK += dS^T Q_scaled      (:1294-1343)
// Every output tile has a single owner: no atomics, fixed summation order.
#pragma once

#include "ct_attn_kernels.hip.h"
#include "ct_lanes.hip.h"

namespace ct {

// ---------------------------------------------------------------------------
// The form of dQ by the number of dS blocks (kDqRecomputes)
// ---------------------------------------------------------------------------
// dS blocks of one query head, all batch rows. (Per row: where the last key block's start and how many it has.)
CT_DEVICE int ds_blocks_per_head(const AttnParams& p) {
  const int nrb = p.S / 32;
  int blocks = 0;
  for (int b = lane_id(); b < p.B; b += 64) {
    const int* last = p.meta + ((size_t)b * nrb + nrb - 1) * kMetaW;
    blocks += last[kDsOff] + max(last[kQLast] - last[kQFirst] + 1, 0);
  }
  return lane_value(wave_scan(blocks), 63);
}
CT_DEVICE bool dq_recomputes(const AttnParams& p) { return uniform(meta_const(p.dkv_header)[kDqRecomputes]) != 0; }
CT_DEVICE void leave_dkv_choice(const AttnParams& p) {
  if (!p.wide_least_blocks || threadIdx.x >= 64) return;
  const int blocks = ds_blocks_per_head(p);
  if (threadIdx.x == 0) p.dkv_header[kDkvWide] = blocks >= p.wide_least_blocks;
}
// Whether this launch's dK/dV kernel is not the one that the documents call for.
CT_DEVICE bool other_dkv_kernel(const AttnParams& p, bool wide) {
  return p.dkv_by_blocks && (uniform(p.dkv_header[kDkvWide]) != 0) != wide;
}

// ---------------------------------------------------------------------------
// dQ
// ---------------------------------------------------------------------------
// The dK/dV kernels work on unscaled Q K^T and put the softmax scale into the exponent. Any finite
// scale is legal (the operator only asks for a finite one): a scale too small for lse / scale to
// stay finite (|scale| < 1e-30, zero included) is replaced there by 1e-30, for which scale * S
// vanishes against lse in f32 all the same (dK is still multiplied by the true scale), and a
// masked pair is marked by the infinity that the sign of the exponent's scale turns into -inf.
__host__ __device__ inline float exponent_scale(float scale) {
  return (scale < 1e-30f && scale > -1e-30f) ? 1e-30f : scale;
}
CT_DEVICE float masked_score(float scale) { return exponent_scale(scale) < 0.f ? -kNegInf : kNegInf; }

// P = exp2(S log2e - lse2), dS = P (dP - delta) for one 32-key block, in place in s.
CT_DEVICE void dq_arith(f32x16& s, const f32x16& dp, float lse2, float delta_q) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float prob = exp2_fast(fmaf(s[r], kLog2e, -lse2));
    s[r] = prob * (dp[r] - delta_q);
  }
}

// The same for dp = dP - delta.
CT_DEVICE void dq_arith(f32x16& s, const f32x16& dp, float lse2) {
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = exp2_fast(fmaf(s[r], kLog2e, -lse2)) * dp[r];
}

// What a key tile of the dQ kernel for D = 128 needs besides its sums, the same for every tile.
struct DqFrame {
  const RowFragOffsets<16>& ro;
  const TrFragOffsets<16, KSlots::kAccum>& to;
  const bf16x8* qf;     // Q and dO fragments
  const bf16x8* dof;
  float lse2, delta;    // of the lane's query row
};

// One key tile as one generated stream (gen_attn_asm.py). MASKED: bit e of `allowed` tells whether the pair of element e is
// allowed (key 8 (e / 4) + 4 half + e % 4 of the tile).
template <int STAGE_OFF, bool MASKED>
CT_DEVICE void dq_step_128(const DqFrame& f, unsigned allowed) {
#define CT_DQ_STEP_OPERANDS                                                                                             \
  "v"(f.qf[0]), "v"(f.qf[1]), "v"(f.qf[2]), "v"(f.qf[3]), "v"(f.qf[4]), "v"(f.qf[5]), "v"(f.qf[6]), "v"(f.qf[7]),       \
      "v"(f.dof[0]), "v"(f.dof[1]), "v"(f.dof[2]), "v"(f.dof[3]), "v"(f.dof[4]), "v"(f.dof[5]), "v"(f.dof[6]),          \
      "v"(f.dof[7]), "v"(f.ro.ptr[0]), "v"(f.ro.ptr[1]), "v"(f.ro.ptr[2]), "v"(f.ro.ptr[3]), "v"(f.ro.ptr[4]),          \
      "v"(f.ro.ptr[5]), "v"(f.ro.ptr[6]), "v"(f.ro.ptr[7]), "v"(f.to.ptr[0][0]), "v"(f.to.ptr[0][1]),                   \
      "v"(f.to.ptr[0][2]), "v"(f.to.ptr[0][3]), "v"(f.to.ptr[1][0]), "v"(f.to.ptr[1][1]), "v"(f.to.ptr[1][2]),          \
      "v"(f.to.ptr[1][3]), "v"(f.lse2), "v"(f.delta), "s"(kLog2e), "i"(STAGE_OFF)
  if constexpr (MASKED)
    asm volatile(CT_DQ_STEP_MASKED_SEQUENCE
                 : : CT_DQ_STEP_OPERANDS, "v"(allowed), "s"(kNegInf)
                 : "memory", CT_DQ_STEP_SCRATCH, CT_DQ_ACCUMULATORS);
  else
    asm volatile(CT_DQ_STEP_SEQUENCE : : CT_DQ_STEP_OPERANDS : "memory", CT_DQ_STEP_SCRATCH, CT_DQ_ACCUMULATORS);
#undef CT_DQ_STEP_OPERANDS
}

// The pairs of a tile whose key has the row's id, and those whose key is not behind `last_rel` (of the lane's half).
template <int STAGE_OFF>
CT_DEVICE unsigned dq_pairs_of_id(lds_addr ids, int id) {
  unsigned allowed;
  asm volatile(CT_DQ_IDS_SEQUENCE
               : "=&v"(allowed) : "v"(ids), "v"(id), "i"(STAGE_OFF)
               : "memory", CT_MASK_PAIRS, CT_DQ_STEP_SCRATCH, CT_DQ_ACCUMULATORS);
  return allowed;
}
CT_DEVICE unsigned dq_pairs_up_to(int last_rel) {
  const int count = min(max(last_rel >> 3, -1) * 4 + min((last_rel & 7) + 1, 4), 32);
  return count <= 0 ? 0u : ~0u >> (32 - count);
}

// One query tile (4 / HS row blocks x HS heads of one KV head), start to finish. STATS: with the rows' statistics, which are
// there already otherwise.
template <int D, int HS, int PER_UNIT, bool STATS>
CT_DEVICE void attn_dq_item(const AttnParams& p, int b, int kvh, int slice, int qt, const lds_addr lds_base) {
  constexpr int kStage = KvStage<D>::kBytes;
  // (the fragment pointers are rebuilt per item from an opaque base: kept across the item loop
  // they end up spilled and reloaded in the key-tile loop)
  lds_addr lds0 = lds_base;
  asm volatile("" : "+v"(lds0));
  // (and for D = 128, whose item loop has no room for their shares of the lane either, from an opaque lane)
  RowFragOffsets<D / 8> ro(lds0);
  TrFragOffsets<D / 8, KSlots::kAccum> to(lds0);
  if constexpr (D == 128) {
    const int lane = lane_id_here();
    ro = RowFragOffsets<D / 8>(lds0, lane);
    to = TrFragOffsets<D / 8, KSlots::kAccum>(lds0, lane);
  }

  const QueryTileContext<D, HS> ctx(p, b, kvh, slice, qt);
  const int l = lane_id(), half = l >> 5, w = threadIdx.x >> 6;
  const size_t q_row_stride = (size_t)p.Hq * D;
  const size_t kv_row_stride = (size_t)p.Hkv * D;
  const size_t stat_t = ((size_t)ctx.work.b * p.Hq + ctx.work.h) * p.S + ctx.pos;  // head-major
  const float lse2 = p.lse[ctx.stat_off] * kLog2e;
  float minus_delta_q = STATS ? 0.f : p.delta[stat_t];

  // The first key tile's copies go first (stage 0), the rows of Q, dO and O behind them; their
  // way into fragments leads through this wavefront's patch in stage 1, which nothing uses yet.
  int t = ctx.first;
  const bool any_tile = t <= ctx.last;
  KvCursor<D> next(ctx.kbase, ctx.vbase, ctx.segb, kv_row_stride, any_tile ? t : 0);
  KeyTileBounds kb = {0, 0, 0};
  if (any_tile) {
    next.issue(lds_base);
    kb = key_tile_bounds(ctx.meta_b, t);
  }
  bf16x8 qf[D / 16], dof[D / 16];
  u32x4 of[D / 16];  // this row's half of `out`, for delta
  {
    const size_t block_off = (((size_t)ctx.work.b * p.S + ctx.work.rb * 32) * p.Hq + ctx.work.h) * D;
    const lds_addr patch = lds0 + kStage + uniform(w) * 32 * D * 2;
    RowBlockLoader<D> q_rows, do_rows, o_rows;
    q_rows.request(p.q + block_off, q_row_stride);
    do_rows.request(p.dout + block_off, q_row_stride);
    if constexpr (STATS) o_rows.request(p.out + block_off, q_row_stride);
    q_rows.to_fragments(patch, qf);
    do_rows.to_fragments(patch, dof);
    if constexpr (STATS) o_rows.to_fragments(patch, of);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) qf[ks] = scale_bf16x8(qf[ks], p.scale);
  }
  f32x16 dqacc[D / 32];  // (D = 128: in accumulation registers)
  if constexpr (D == 128) {
    asm volatile(CT_DQ_ZERO : : : CT_DQ_ACCUMULATORS);
  } else {
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dqacc[db] = zero16();
  }
  dma_wait_all();
  __syncthreads();

  // delta = sum_d out[row, d] * dout[row, d], after the wait above so that the first key tile's
  // copies are not held back behind these loads; the dK/dV kernel, launched after this one, reads
  // delta and lse * log2(e) head-major
  if constexpr (STATS) {
    float delta_part = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      u32x4 o_bits = of[ks];
      asm volatile("" : "+v"(o_bits));
      const u32x4 do_bits = __builtin_bit_cast(u32x4, dof[ks]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        delta_part = fmaf(__uint_as_float(o_bits[e] << 16), __uint_as_float(do_bits[e] << 16), delta_part);
        delta_part = fmaf(__uint_as_float(o_bits[e] & 0xffff0000u), __uint_as_float(do_bits[e] & 0xffff0000u),
                          delta_part);
      }
    }
    minus_delta_q = -pair_sum(delta_part);
  }
  const float delta_q = -minus_delta_q;
  f32x16 minus_delta;
  if constexpr (D == 64) {
#pragma unroll
    for (int r = 0; r < 16; ++r) minus_delta[r] = -delta_q;
    asm volatile("" : "+v"(minus_delta));
  }
  if (STATS && ctx.active && half == 0) {
    // for the dK/dV kernel: the values it adds to its S and dP blocks, P = exp2((S - lse / scale) *
    // scale * log2(e)) and dS = P (dP - delta)
    p.delta[stat_t] = -delta_q;
    p.lse2[stat_t] = -p.lse[ctx.stat_off] / exponent_scale(p.scale);
  }

  auto step = [&](auto stage_tag) {
    constexpr int CUR = decltype(stage_tag)::value;
    const lds_addr stage = lds0 + CUR * kStage;
    if (t + 1 <= ctx.last) {
      next.advance();
      next.issue(lds_base + (CUR ^ 1) * kStage);
    }
    // (requested behind the products of D = 64: a wait for LDS reads is one for all scalar loads too)
    KeyTileRecords ahead;
    const auto request = [&]() { ahead = KeyTileRecords(ctx.meta_b, min(t + 1, ctx.last)); };
    const bool visits = ctx.wave_visits(kb, t);
    if (D != 64 || !visits) request();
    if (visits) {
      // Same specialisation as the forward: masked scores become -inf, so their
      // probability exp2(-inf) is exactly 0 and so is dS.
      const int k_uniform = uniform(kb.uniform);
      const bool need_seg = ctx.mine.uniform == 0 || ctx.mine.uniform != k_uniform;
      const bool need_causal = t * kKeyTile + kKeyTile - 1 > ctx.mine.end_min;
      const int seg_cmp = ctx.row_valid() ? ctx.seg_q : -1;
      int last_rel = ctx.end_q - t * kKeyTile - 4 * half;
      if (k_uniform != 0 && seg_cmp != k_uniform) last_rel = -1;
      constexpr int kOff = CUR * kStage + KvStage<D>::kK, vOff = CUR * kStage + KvStage<D>::kV;
      if constexpr (D == 128) {
        const DqFrame f{ro, to, qf, dof, lse2, delta_q};
        if (need_seg || need_causal) {
          unsigned allowed = dq_pairs_up_to(last_rel);
          if (k_uniform == 0) allowed &= dq_pairs_of_id<CUR * kStage>(lds0 + KvStage<D>::kSeg + 16 * half, seg_cmp);
          dq_step_128<CUR * kStage, true>(f, allowed);
        } else {
          dq_step_128<CUR * kStage, false>(f, 0);
        }
      } else {
        // Both 32-key blocks at once, or one after the other where registers are for three workgroups on a compute unit.
        // (dP starts from -delta, a register block of its own, and needs no subtraction)
        constexpr int kSteps = D / 16, kBlocks = D / 32, N = PER_UNIT == 2 ? 2 : 1;
        auto blocks = [&](auto first_tag) {
          constexpr int FIRST = decltype(first_tag)::value;
          f32x16 s[N], dp[N];
          fragments_ahead<2 * N * kSteps, N == 2 ? 6 : 4>(
              [&](int i) { return ro.load(i < N * kSteps ? kOff : vOff, FIRST + i % N, i / N % kSteps); },
              [&](int i, bf16x8 keys) {
                const int kb = i % N, ks = i / N % kSteps;
                if (i < N * kSteps) s[kb] = mfma32(keys, qf[ks], ks ? s[kb] : zero16());
                else dp[kb] = mfma32(keys, dof[ks], ks ? dp[kb] : minus_delta);
              });
          if constexpr (FIRST == 0) request();
          if (need_seg || need_causal) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
              if (k_uniform == 0) mask_block_t<true, true>(stage + KvStage<D>::kSeg, seg_cmp, last_rel, FIRST + i, s[i]);
              else mask_block_t<false, true>(stage, seg_cmp, last_rel, FIRST + i, s[i]);
            }
          }
          bf16x8 ds[2 * N];
#pragma unroll
          for (int i = 0; i < N; ++i) dq_arith(s[i], dp[i], lse2);
#pragma unroll
          for (int i = 0; i < 2 * N; ++i) ds[i] = pack_acc8(s[i >> 1], i & 1);
          fragments_ahead<2 * N * kBlocks, 4>([&](int i) { return to.load(kOff, 2 * FIRST + i / kBlocks, i % kBlocks); },
                                              [&](int i, bf16x8 keys) {
                                                dqacc[i % kBlocks] = mfma32(keys, ds[i / kBlocks], dqacc[i % kBlocks]);
                                              });
        };
        blocks(std::integral_constant<int, 0>{});
        if constexpr (N == 1) blocks(std::integral_constant<int, 1>{});
      }
    }
    ahead.pin();
    dma_wait_all();
    __syncthreads();
    kb = ahead.bounds();
    ++t;
  };
  while (t <= ctx.last) {
    step(std::integral_constant<int, 0>{});
    if (t > ctx.last) break;
    step(std::integral_constant<int, 1>{});
  }

  if (ctx.active) {
    const lds_addr patch = lds0 + w * 32 * D * 2;
    bf16* gbase = p.dq + (((size_t)ctx.work.b * p.S + ctx.work.rb * 32) * p.Hq + ctx.work.h) * D;
    if constexpr (D == 128) {
      asm volatile("s_nop 15\n\ts_nop 7" : : : "memory");  // the last sums leave the matrix pipe
      fwd_store_rows(p.scale, patch, gbase, q_row_stride);
    } else {
      store_rows_t<D>(dqacc, p.scale, patch, gbase, q_row_stride);
    }
  }
  // the store patches overlap the stages of the next item: its copies may start once every
  // wavefront has read its patch back
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __syncthreads();
}

// Workgroups of one (head slice, KV head) group share a work counter and pull query tiles of PB
// row blocks from the work-sorted schedules of the batch rows (tile `rank` of row b at pull
// B * rank + b: heaviest tiles first), so a workgroup that drew light tiles simply draws more of
// them. (Static bins left 15 % of the workgroup slots idle at the end of the launch: the time
// of a tile depends on its mix of masked and unmasked key tiles, not just on their number.)
// The group is the fast index of blockIdx: a group stays on one XCD and its K / V rows in that
// XCD's L2. With more groups than counters (kDqCounters) the tiles are dealt round robin.
//
// PER_UNIT workgroups on a compute unit: at head dimension 64 two, or for large launches three (168 registers: the wavefronts
// of a SIMD wait less for each other's products, but each takes a tile's two blocks one after the other and has more to do per
// query tile). dQ, us, two / three: [1, 25472, 64/8 heads of 64], images, 1289 / 1186; [6, 2816, 64/16], images, 692 / 642; [4, 4096, 64/8]
// 374 / 342; [4, 4992, 48/8], documents of 99 to 152, 160 / 151. Below 12288 row blocks short documents lose more than long ones
// gain: [4, 5376, 16/16], 10752, 45 to 111, 74 / 81, [1, 17280, 12/4], 6480, 121 to 236, 49 / 55, [1, 16384, 16/2], whole rows, 813 / 752.
template <int D, int HS, int PER_UNIT, bool STATS>
CT_DEVICE void attn_dq_tiles(const AttnParams& p, int index, int workgroups, const lds_addr lds0, int* next_pull) {
  constexpr int PB = 4 / HS;
  const int nrb = p.S / 32;
  const int slices = (p.Hq / p.Hkv) / HS;
  const int groups = slices * p.kvh_count;
  const int group = index % groups, member = index / groups, members = workgroups / groups;
  const int kvh = p.kvh_base + group % p.kvh_count, slice = group / p.kvh_count;
  const int tpr = bin_tiles_per_row(nrb, PB);
  const int total = p.B * tpr;
  const MetaPtr sched = meta_const(p.sched + query_schedule_offset(nrb, PB));
  const bool dynamic = slices * p.Hkv <= kDqCounters;
  if (!dynamic && member >= members) return;
  for (int pull = member;; pull += members) {
    if (dynamic) {
      if (threadIdx.x == 0) *next_pull = atomicAdd(&p.dq_counters[slice * p.Hkv + kvh], 1);
      __syncthreads();
      pull = uniform(*next_pull);
      __syncthreads();
    }
    if (pull >= total) break;
    const int b = pull % p.B, rank = pull / p.B;
    const int qt = uniform(sched[(size_t)b * schedule_ints(nrb) + rank]);
    attn_dq_item<D, HS, PER_UNIT, STATS>(p, b, kvh, slice, qt, lds0);
  }
}
template <int D, int HS, int PER_UNIT>
__global__ __launch_bounds__(256, PER_UNIT) void attn_dq_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  if (D == 64 && p.ds_most_blocks && !dq_recomputes(p)) return;
  __shared__ int next_pull;
  attn_dq_tiles<D, HS, PER_UNIT, true>(p, blockIdx.x, gridDim.x, lds_address_of(smem_raw), &next_pull);
}

// ---------------------------------------------------------------------------
// dK / dV
// ---------------------------------------------------------------------------
constexpr int kQueryTile = 32;

// LDS stage: Q tile, dO tile (32 x D bf16 each), then lse2 / delta (f32) and
// seg / end (i32), 32 entries each.
template <int D>
struct QdoStage {
  static constexpr int kTileBytes = kQueryTile * D * 2;
  static constexpr int kQ = 0;
  static constexpr int kDo = kTileBytes;
  static constexpr int kLse = 2 * kTileBytes;
  static constexpr int kDelta = kLse + kQueryTile * 4;
  static constexpr int kSeg = kDelta + kQueryTile * 4;
  static constexpr int kEnd = kSeg + kQueryTile * 4;
  static constexpr int kBytes = kEnd + kQueryTile * 4;
  static constexpr int kPatchBytes = 4 * 32 * D * 2;
  // resident V rows of the workgroup's 128 keys (32 per wavefront), after the two stages
  static constexpr int kVResident = 2 * kBytes;
  static constexpr int kTotalBytes = 2 * kBytes + kPatchBytes;
};

// The walk of a dK/dV workgroup over its (head, query block) items, query block fastest, as the addresses that
// move with it: the rows of Q and dO, the statistics this wavefront fetches and the block's bounds. A step adds a
// constant, the one of a next query block or the one of a next head's first block. (Formed from the coordinates
// for every item, the same addresses were 64-bit products and a chain of branches over the statistics array,
// about 60 scalar instructions a step of 300.)
//
// The four statistics arrays (lse2, delta: head-major f32; segment ids, visible ends: i32) are 128 contiguous
// bytes each for the 32 rows and sit in the stage in that order; wavefront w fetches array w with its first 8
// lanes, one copy instruction. Without visible ends (plain causal) wavefront 3 fetches nothing.
template <int D>
struct QdoCursor {
  int head, left;  // left: query blocks of this head behind this one
  const char* q;
  const char* dout;
  const char* stat;
  const char* bounds;
  long long row_step, row_wrap, stat_wrap, bounds_wrap;
  unsigned long long stat_lanes;

  CT_DEVICE QdoCursor(const AttnParams& p, int b, int head_, int qb, int q_lo, int q_hi, int which) : head(head_), left(q_hi - qb) {
    const size_t origin = (((size_t)b * p.S + qb * kQueryTile) * p.Hq + head) * D * sizeof(bf16);
    q = reinterpret_cast<const char*>(p.q) + origin;
    dout = reinterpret_cast<const char*>(p.dout) + origin;
    bounds = reinterpret_cast<const char*>(p.meta) + ((size_t)b * (p.S / 32) + qb) * (kMetaW * sizeof(int));
    const bool head_major = which < 2;
    const size_t row = (head_major ? (size_t)b * p.Hq + head : (size_t)b) * p.S + qb * kQueryTile;
    const char* array = which == 0   ? reinterpret_cast<const char*>(p.lse2)
                        : which == 1 ? reinterpret_cast<const char*>(p.delta)
                        : which == 2 ? reinterpret_cast<const char*>(p.seg)
                                     : reinterpret_cast<const char*>(p.end);
    stat = array + row * 4;
    stat_lanes = which == 3 && !p.end ? 0 : 0xff;
    const long long back = q_hi - q_lo;  // from the last query block of a head to its first
    row_step = (long long)kQueryTile * p.Hq * D * (long long)sizeof(bf16);
    row_wrap = D * (long long)sizeof(bf16) - back * row_step;
    stat_wrap = (head_major ? (long long)p.S * 4 : 0) - back * (kQueryTile * 4);
    bounds_wrap = -back * (long long)(kMetaW * sizeof(int));
  }
  CT_DEVICE void advance(int blocks) {
    const bool wrap = left == 0;
    const long long rows = wrap ? row_wrap : row_step;
    q += rows;
    dout += rows;
    stat += wrap ? stat_wrap : (long long)(kQueryTile * 4);
    bounds += wrap ? bounds_wrap : (long long)(kMetaW * sizeof(int));
    left = wrap ? blocks - 1 : left - 1;
    head += wrap ? 1 : 0;
  }
  // asynchronous copy of the item into `stage`
  CT_DEVICE void fetch(const TileDma<kQueryTile, D / 8>& dma, lds_addr stage, int wave) const {
    dma.issue(q, stage + QdoStage<D>::kQ, wave);
    dma.issue(dout, stage + QdoStage<D>::kDo, wave);
    dma16_lanes_s(stat, (unsigned)lane_id_here() * 16, stage + QdoStage<D>::kLse + wave * (kQueryTile * 4), stat_lanes);
  }
  CT_DEVICE QueryBlockBounds query_bounds() const { return query_block_bounds(reinterpret_cast<const int*>(bounds), 0); }
};

// What a step of the dK/dV kernel for D = 128 needs besides its sums, the same in every step.
struct DkvFrame {
  const RowFragOffsets<16>& ro;
  const TrFragOffsets<16, KSlots::kAccum>& to;
  const bf16x8* kf;     // K fragments
  lds_addr stat_ptr;    // LDS base + 16 * (lane / 32)
  float scale_log2e;
  unsigned v_off;       // byte offset of this wavefront's V rows
};

// Which pairs of a step are allowed: all, those with the key's id and a key not behind the row's visible end, or those with
// its id and a key not behind the row itself.
enum class DkvPairs { kAll, kToEnds, kToRows };

// One step as one generated stream (gen_attn_asm.py). `key`: for kToRows relative to the first query row of the lane's
// half. STORE: the dS block leaves to `block` as well, as the lanes hold it: two runs of 64 x 16 bytes.
template <int STAGE_OFF, DkvPairs PAIRS, bool STORE>
CT_DEVICE void dkv_step_128(const DkvFrame& f, float masked, int id, int key, char* block, unsigned lane16) {
#define CT_DKV_STEP_OPERANDS                                                                                            \
  "v"(f.kf[0]), "v"(f.kf[1]), "v"(f.kf[2]), "v"(f.kf[3]), "v"(f.kf[4]), "v"(f.kf[5]), "v"(f.kf[6]), "v"(f.kf[7]),       \
      "v"(f.ro.ptr[0]), "v"(f.ro.ptr[1]), "v"(f.ro.ptr[2]), "v"(f.ro.ptr[3]), "v"(f.ro.ptr[4]), "v"(f.ro.ptr[5]),       \
      "v"(f.ro.ptr[6]), "v"(f.ro.ptr[7]), "v"(f.to.ptr[0][0]), "v"(f.to.ptr[0][1]), "v"(f.to.ptr[0][2]),                \
      "v"(f.to.ptr[0][3]), "v"(f.to.ptr[1][0]), "v"(f.to.ptr[1][1]), "v"(f.to.ptr[1][2]), "v"(f.to.ptr[1][3]),          \
      "v"(f.stat_ptr), "s"(f.scale_log2e), "s"(f.v_off), "i"(STAGE_OFF)
#define CT_DKV_STEP_CLOBBERS "memory", "vcc", "scc", "s96", "s97", CT_DKV_STEP_SCRATCH, CT_DKV_ACCUMULATORS
#define CT_DKV_STEP(SEQUENCE, ...) asm volatile(SEQUENCE : : CT_DKV_STEP_OPERANDS, ##__VA_ARGS__ : CT_DKV_STEP_CLOBBERS)
#define CT_DKV_MASK "s"(masked), "v"(id), "v"(key)
#define CT_DKV_STORE "s"(block), "v"(lane16)
  if constexpr (PAIRS == DkvPairs::kAll) {
    if constexpr (STORE) CT_DKV_STEP(CT_DKV_STEP_STORE_SEQUENCE, CT_DKV_STORE);
    else CT_DKV_STEP(CT_DKV_STEP_SEQUENCE);
  } else if constexpr (PAIRS == DkvPairs::kToEnds) {
    if constexpr (STORE) CT_DKV_STEP(CT_DKV_STEP_ENDS_STORE_SEQUENCE, CT_DKV_MASK, CT_DKV_STORE);
    else CT_DKV_STEP(CT_DKV_STEP_ENDS_SEQUENCE, CT_DKV_MASK);
  } else {
    if constexpr (STORE) CT_DKV_STEP(CT_DKV_STEP_ROWS_STORE_SEQUENCE, CT_DKV_MASK, CT_DKV_STORE);
    else CT_DKV_STEP(CT_DKV_STEP_ROWS_SEQUENCE, CT_DKV_MASK);
  }
#undef CT_DKV_STORE
#undef CT_DKV_MASK
#undef CT_DKV_STEP
#undef CT_DKV_STEP_CLOBBERS
#undef CT_DKV_STEP_OPERANDS
}

// The rows of 32 keys of D = 128 on their way through a wavefront's patch (swizzled tile layout): element r of column block
// db is row 8 (r / 4) + 4 half + r % 4, chunk 4 db + j / 8, and lies a constant behind one of two addresses. (Formed from row
// and chunk numbers for each, they were much of the end of a tile: documents of 17 to 113 in [1, 2048, 8/8 heads], the kernel
// 20.6 us with them, 19.5 without.)
struct KeyRowsPatch {
  lds_addr at[2];
  CT_DEVICE KeyRowsPatch(lds_addr patch, int l) {
    const int j = l & 31, half = l >> 5;
#pragma unroll
    for (int odd = 0; odd < 2; ++odd) at[odd] = patch + half * 1024 + (j & 7) * 2 + (((j >> 3) ^ half ^ (2 * odd)) << 4);
  }
  CT_DEVICE void store(int db, const f32x16& sum) const {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      lds_store<bf16>(at[r / 4 % 2] + (2048 * (r / 4) + 256 * (r % 4) + 64 * (db ^ (r % 4))), (bf16)sum[r]);
  }
};

// Store a (32 rows x D) accumulator (lanes along D) as bf16 rows via an LDS patch. (Head dimension 64 with two addresses
// as well: what the compiler then does with the item loop in front takes 1 to 2 % longer.)
template <int D>
CT_DEVICE void store_rows(const f32x16* acc, lds_addr patch, bf16* gbase, size_t row_stride) {
  constexpr int CPR = D / 8;
  const int l = lane_id(), j = l & 31, half = l >> 5;
  if constexpr (D == 128) {
    const KeyRowsPatch rows(patch, l);
#pragma unroll
    for (int db = 0; db < 4; ++db) rows.store(db, acc[db]);
    __builtin_amdgcn_wave_barrier();
    PatchRows<D>::to_global(patch, l, gbase, row_stride);
    return;
  }
#pragma unroll
  for (int db = 0; db < D / 32; ++db) {
    const int col = db * 32 + j;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      lds_store<bf16>(patch + tile_byte_offset<CPR>(acc_row(r, half), col >> 3) + (col & 7) * 2,
                      (bf16)acc[db][r]);
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int n = 0; n < 32 * CPR / 64; ++n) {
    const int e = l + 64 * n;
    const int row = e / CPR, c = e % CPR;
    const u32x4 val = lds_load<u32x4>(patch + tile_byte_offset<CPR>(row, c));
    store_global16(gbase + (size_t)row * row_stride + c * 8, val);
  }
}

// An accumulator that only the assembly statements name, a[16 INDEX : 16 INDEX + 15]. A store in front may still read the
// registers that the statement writes, and the compiler does not wait for it here.
template <int INDEX>
CT_DEVICE f32x16 read_accumulator() {
  float v[16];
  asm volatile("s_nop 1\n\t" CT_DKVW_READ
               : "=v"(v[0]), "=v"(v[1]), "=v"(v[2]), "=v"(v[3]), "=v"(v[4]), "=v"(v[5]), "=v"(v[6]), "=v"(v[7]),
                 "=v"(v[8]), "=v"(v[9]), "=v"(v[10]), "=v"(v[11]), "=v"(v[12]), "=v"(v[13]), "=v"(v[14]), "=v"(v[15])
               : "i"(16 * INDEX));
  f32x16 out;
#pragma unroll
  for (int e = 0; e < 16; ++e) out[e] = v[e];
  return out;
}

// dK or dV of a wavefront's 32 keys of D = 128, accumulators FIRST to FIRST + 3, as bf16 rows (store_rows), or to `mine` as
// the f32 sums of a chunk. One accumulator at a time: what the compiler has no room for it would put into accumulation
// registers.
template <int FIRST, bool SCALED>
CT_DEVICE void leave_accumulators(float scale, float* mine, lds_addr patch, bf16* gbase, size_t row_stride) {
  const int l = lane_id_here();
  const KeyRowsPatch rows(patch, l);
  const auto each = [&](auto db_tag) {
    constexpr int kDb = decltype(db_tag)::value;
    f32x16 sum = read_accumulator<FIRST + kDb>();
    if (SCALED) {
#pragma unroll
      for (int e = 0; e < 16; ++e) sum[e] *= scale;
    }
    if (mine) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        f32x4 quad;
#pragma unroll
        for (int e = 0; e < 4; ++e) quad[e] = sum[4 * q4 + e];
        *reinterpret_cast<f32x4*>(mine + l * 4 + (kDb * 4 + q4) * 256) = quad;
      }
    } else {
      rows.store(kDb, sum);
    }
  };
  each(std::integral_constant<int, 0>{});
  each(std::integral_constant<int, 1>{});
  each(std::integral_constant<int, 2>{});
  each(std::integral_constant<int, 3>{});
  if (mine) return;
  __builtin_amdgcn_wave_barrier();
  PatchRows<128>::to_global(patch, l, gbase, row_stride);
  __builtin_amdgcn_wave_barrier();  // (the other tensor leaves through the same patch)
}

// Number of (head, query block) items of 128-key tile `tile` (= batch row * tiles per row + kt).
CT_DEVICE int dkv_tile_items(const int* meta, int nrb, int tile, int g, int* q_lo_out = nullptr) {
  const int nt = nrb / 4;
  const int* m = meta + ((size_t)(tile / nt) * nrb + (size_t)(tile % nt) * 4) * kMetaW;
  int q_lo = INT_MAX, q_hi = -1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    q_lo = min(q_lo, m[i * kMetaW + kQFirst]);
    q_hi = max(q_hi, m[i * kMetaW + kQLast]);
  }
  if (q_lo_out) *q_lo_out = q_lo;
  return q_lo <= q_hi ? (q_hi - q_lo + 1) * g : 0;
}

CT_DEVICE int dkv_split_count(int items, int target) {
  return items <= target ? 1 : min(kDkvMaxSplit, (items + target - 1) / target);
}

// Builds the dK/dV work list (one workgroup of 1024 threads): chunk target from
// the total amount of work, chunk count per tile, entries bucketed by
// decreasing work. Clears the dQ kernel's work counters.
template <int D>
CT_DEVICE void dkv_schedule(const int* meta, int B, int S, int Hkv, int g, int max_entries, int max_partials, int* header,
                            int2* entries, int* zeroed, int zeroed_count) {
  for (int i = threadIdx.x; i < zeroed_count; i += 1024) zeroed[i] = 0;  // dQ's work counters
  __shared__ int red[32];  // one value per wavefront, or two
  __shared__ int hist[256];
  __shared__ int fill[256];
  __shared__ int carry;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int nrb = S / 32, ntiles = B * (nrb / 4);

  // Reductions and scans run inside the wavefronts (lane moves) and meet once in LDS: the
  // kernel is one workgroup on an otherwise idle GPU, so its time is its chain of barriers.
  auto block_sums = [&](int u, int v, int* sum_u, int* sum_v) {
    const int wave_u = lane_value(wave_scan(u), 63), wave_v = lane_value(wave_scan(v), 63);
    if (lane == 0) {
      red[wave] = wave_u;
      red[16 + wave] = wave_v;
    }
    __syncthreads();
    const int sums = wave_scan(lane < 32 ? red[lane] : 0);
    __syncthreads();
    *sum_u = lane_value(sums, 15);
    *sum_v = lane_value(sums, 31) - *sum_u;
  };
  auto block_max = [&](int v) {
    const int most = lane_value(wave_scan<true>(v), 63);
    if (lane == 0) red[wave] = most;
    __syncthreads();
    const int out = lane_value(wave_scan<true>(lane < 16 ? red[lane] : 0), 15);
    __syncthreads();
    return out;
  };
  // exclusive prefix of v over the workgroup's threads, and the total
  auto block_scan = [&](int v, int* total) {
    const int inc = wave_scan(v);
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    const int sums = wave_scan(lane < 16 ? red[lane] : 0);
    __syncthreads();
    *total = lane_value(sums, 15);
    return (wave ? lane_value(sums, wave - 1) : 0) + inc - v;
  };
  // this thread's first tile is read once; further tiles (more than 1024) are re-read per pass
  const int items_first = tid < ntiles ? dkv_tile_items(meta, nrb, tid, g) : 0;
  auto items_of = [&](int t) { return t == tid ? items_first : dkv_tile_items(meta, nrb, t, g); };

  long long local = 0;
  for (int t = tid; t < ntiles; t += 1024) local += items_of(t);
  // (the threads' sums in halves: both fit in 32 bits over 1024 threads with up to 8192 tiles each)
  int high = 0, low = 0;
  block_sums((int)(local >> 16), (int)(local & 0xffff), &high, &low);
  const long long total = ((long long)high << 16) + low;
  long long want = (total * Hkv + kDkvSlots - 1) / kDkvSlots;  // one compute slot's fair share
  const long long pairs = (long long)ntiles * Hkv;  // (key tile, KV head)
  const int least = pairs <= kDkvSlots / 16 ? kDkvMinChunk / 4 : pairs <= kDkvSlots / 2 ? kDkvMinChunk / 2 : kDkvMinChunk;
  // With more tiles than slots a chunk may be longer than the share: what it is over, it walks alone on its compute unit, at nearly
  // twice the pace, and a cut costs a way into another walk and 131 KB of sums written, read and added, as much as some items do.
  // So short shares are cut at 1.4 of them. dK/dV and dQ with the sums of [B, S, heads of 128], us, cut by the share / so:
  // [8, 2048, 8/8], documents of 64 to 2048 (a share of 22 items), 129 / 118; [6, 1024, 48/16], 392 to 424 (34), 152 / 130; [2, 2304,
  // 16/16], images (33), 162 / 132; [4, 6272, 8/4], 407 to 3607 (96), 346 / 331; 38 drawn calls with cuts and shares of up to 128
  // items 0.993 to 1.23, 1.037 in the geometric mean. Beyond, where the sums weigh less than a tail of one chunk in a second round,
  // 0.895 ([3, 5760, 16/4], images) to 1.045. At head dimension 64, whose sums are half as long, 0.91 to 1.02 (19 calls).
  if (D == 128 && pairs > kDkvSlots && want <= 128) want += want * 2 / 5;
  int target = (int)min((long long)INT_MAX / 2, max((long long)least, want));

  // Where there are somewhat fewer tiles than slots the share is not always the best target: 432 tiles of 1.2 shares cut in two
  // take two rounds of the slots, as long as they take whole in one, and leave 80 MB of partial sums to write, read and add. The
  // target is the one of four with the least estimated end, in items: the longest chunk, or where there are more chunks than
  // slots the one that is dealt second to the slot of the slots' shortest (twice its length), and the sums at 0.03 items per
  // partial sum (131 KB written and read, an item 1.8 us). It has to be 8 % better than the share: a workgroup that is left
  // alone on its compute unit at the end is the faster for it. Fewer tiles leave slots idle and are cut by the share, longer
  // lists end evenly; at head dimension 64 shorter chunks gain more than half as large sums cost ([2, 10368, 12/2 of 64],
  // documents of 50 to 414: dK/dV 46 us, by such an estimate 58). The whole pass, us: [3, 4480, 32/4 of 128], documents of
  // 36 to 58, 317 -> 269; [2, 2048, 16/16], images, 222 -> 191; [1, 3456, 64/16], 87 to 178, 210 -> 184; 40 drawn shapes
  // 0.99 to 1.18. (Counted a wavefront at a time: with an atomic per tile and target the list took 6 us more.) The estimate
  // itself takes 2.3 us, and where the share cuts no tile all four targets give one list: it is left out there (the list of
  // [1, 5248, 8/8], documents of 16 to 32, 9.6 -> 7.8 us).
  if (D == 128 && pairs > kDkvSlots / 2 && pairs <= kDkvSlots && __syncthreads_or(items_first > target)) {
    constexpr int kTargets = 4, kBuckets = 256;
    __shared__ int chunks[kTargets * kBuckets];  // by length, the longest in the last one
    __shared__ int split[kTargets], longest[kTargets];
    __shared__ float ends[kTargets];
    const auto candidate = [&](int k) { return (int)min((long long)INT_MAX / 4, (long long)target * (k == 3 ? 8 : 4 + k) / 4); };
    const float bucket_items = (float)candidate(kTargets - 1) / kBuckets;
    for (int i = tid; i < kTargets * kBuckets; i += 1024) chunks[i] = 0;
    if (tid < kTargets) split[tid] = longest[tid] = 0;
    __syncthreads();
    const float buckets_per_item = 1.f / bucket_items;
    if (wave * 64 < ntiles) {  // (at most kDkvSlots tiles: one per thread)
      const int items = tid < ntiles ? items_first : 0;
#pragma unroll
      for (int k = 0; k < kTargets; ++k) {
        const int ns = dkv_split_count(items, candidate(k)), per = (items + ns - 1) / ns;
        if (items) atomicAdd(&chunks[k * kBuckets + min(kBuckets - 1, (int)((float)per * buckets_per_item))], ns);
        const int parts = lane_value(wave_scan(ns > 1 ? ns : 0), 63), most = lane_value(wave_scan<true>(per), 63);
        if (lane == 0) {
          if (parts) atomicAdd(&split[k], parts);
          atomicMax(&longest[k], most);
        }
      }
    }
    __syncthreads();
    if (wave < kTargets) {  // a wavefront per target, four buckets per lane, the longest chunks in lane 0
      int count[4], mine = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) mine += count[j] = chunks[wave * kBuckets + (kBuckets - 1 - 4 * lane - j)];
      const int upto = wave_scan(mine);
      int second = 0;  // bucket of chunk kDkvSlots + 1, where it is one of this lane's
      int before = upto - mine;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool here = (long long)before * Hkv <= kDkvSlots && (long long)(before + count[j]) * Hkv > kDkvSlots;
        before += count[j];
        if (here) second = kBuckets - 4 * lane - j;
      }
      second = lane_value(wave_scan<true>(second), 63);
      const float chunk = (float)longest[wave];
      if (lane == 0) ends[wave] = fmaxf(chunk, 2.f * (float)second * bucket_items) + 0.03f * (float)split[wave] * (float)Hkv;
    }
    __syncthreads();
    float least_end = 0.92f * ends[0];
    int best = target;
#pragma unroll
    for (int k = 1; k < kTargets; ++k)
      if (ends[k] < least_end) {
        least_end = ends[k];
        best = candidate(k);
      }
    target = uniform(best);
  }

  // Entry and partial-slot counts for this target; coarsen the target if they overflow the
  // space the host reserved (cannot happen for target >= want, kept as a guard).
  int max_work = 1;
  for (;;) {
    int entry_count = 0, partial_count = 0, local_max = 1;
    for (int t = tid; t < ntiles; t += 1024) {
      const int items = items_of(t);
      const int ns = dkv_split_count(items, target);
      entry_count += ns;
      partial_count += ns > 1 ? ns : 0;
      local_max = max(local_max, (items + ns - 1) / ns);
    }
    int entries_wanted = 0, partials_wanted = 0;
    block_sums(entry_count, partial_count, &entries_wanted, &partials_wanted);
    max_work = block_max(local_max);
    if (entries_wanted <= max_entries && partials_wanted <= max_partials) break;
    target = target >= INT_MAX / 4 ? INT_MAX / 2 : target * 2;
  }

  // Histogram of entries over 256 buckets of decreasing work.
  if (tid < 256) {
    hist[tid] = 0;
    fill[tid] = 0;
  }
  if (tid == 0) carry = 0;
  __syncthreads();
  auto bucket_of = [&](int work) { return 255 - (int)((long long)work * 255 / max_work); };
  for (int t = tid; t < ntiles; t += 1024) {
    const int items = items_of(t);
    const int ns = dkv_split_count(items, target);
    const int per = (items + ns - 1) / ns, full = min(ns, items / max(per, 1));  // chunks of `per` items; then one of
    const int rest = items - full * per;                                         // the rest, then empty ones
    if (full > 0) atomicAdd(&hist[bucket_of(per)], full);
    if (full < ns) atomicAdd(&hist[bucket_of(rest)], 1);
    if (full + 1 < ns) atomicAdd(&hist[bucket_of(0)], ns - full - 1);
  }
  __syncthreads();
  {
    int entries_total = 0;
    const int start = block_scan(tid < 256 ? hist[tid] : 0, &entries_total);
    if (tid < 256) hist[tid] = start;  // bucket -> first position in the list
    if (tid == 0) {
      header[0] = entries_total;
      header[1] = target;
    }
  }
  __syncthreads();

  // Partial-slot offsets by a running scan over tiles, then scatter.
  for (int base = 0; base < ntiles; base += 1024) {
    const int t = base + tid;
    int items = 0, ns = 1;
    if (t < ntiles) {
      items = items_of(t);
      ns = dkv_split_count(items, target);
    }
    const int mine = (t < ntiles && ns > 1) ? ns : 0;
    int chunk_total = 0;
    const int slot0 = carry + block_scan(mine, &chunk_total);
    __syncthreads();
    if (tid == 0) carry += chunk_total;
    if (t < ntiles) {
      const int per = (items + ns - 1) / ns, full = min(ns, items / max(per, 1)), rest = items - full * per;
      const auto place = [&](int begin, int end, int work) {  // chunks begin .. end - 1
        if (begin >= end) return;
        const int bk = bucket_of(work), pos = hist[bk] + atomicAdd(&fill[bk], end - begin);
        for (int c = begin; c < end; ++c) entries[pos + c - begin] = make_int2(t, c | (ns << 8) | (slot0 << 16));
      };
      place(0, full, per);
      place(full, min(full + 1, ns), rest);
      place(full + 1, ns, 0);
    }
    __syncthreads();
  }
}

template <int D>
__global__ __launch_bounds__(1024) void attn_dkv_schedule_kernel(AttnParams p, int kvh_side_by_side) {
  if (D == 128) leave_dkv_choice(p);
  dkv_schedule<D>(p.meta, p.B, p.S, kvh_side_by_side, p.Hq / p.Hkv, p.dkv_max_entries, p.dkv_max_partials, p.dkv_header,
               p.dkv_entries, p.dq_counters, kDqCounters);
}

// The work list and, in the other workgroups, the row statistics: two independent passes in one launch. The
// list is one workgroup's chain of barriers (7 us at [2, 1024], the statistics 4 us), so the shorter of the
// two costs nothing.
template <int D>
__global__ __launch_bounds__(1024) void attn_bwd_setup_kernel(AttnParams p, int kvh_side_by_side, float exponent_scale) {
  const bool asked = p.ds_most_blocks && (blockIdx.x == 0 || !p.dq_rides);
  const bool recompute = asked && ds_blocks_per_head(p) > p.ds_most_blocks;
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) p.dkv_header[kDqRecomputes] = recompute;
    if (D == 128) leave_dkv_choice(p);
    dkv_schedule<D>(p.meta, p.B, p.S, kvh_side_by_side, p.Hq / p.Hkv, p.dkv_max_entries, p.dkv_max_partials, p.dkv_header,
                 p.dkv_entries, p.dq_counters, kDqCounters);
    return;
  }
  if (recompute) return;  // (that dQ kernel forms the statistics on its way)
  bwd_stats_tiles<D>(p.out, p.dout, p.lse, p.delta, p.lse2, p.B, p.S, p.Hq, exponent_scale,
                     (blockIdx.x - 1) * 4 + (threadIdx.x >> 8), (gridDim.x - 1) * 4, threadIdx.x & 255);
}

// f32 partial sums of one chunk of a split key tile.
template <int D>
struct DkvPartial {
  static constexpr int kPerWave = (D / 32) * 16 * 64;  // floats of one accumulator set of a wavefront
  static constexpr int kPerTensor = 4 * kPerWave;      // dK (or dV) of the 4 wavefronts
  static constexpr size_t kPerChunk = 2 * kPerTensor;
};
template <int D>
CT_DEVICE size_t dkv_partial_offset(int slot, int Hkv, int kvh, int wave) {
  return ((size_t)slot * Hkv + kvh) * DkvPartial<D>::kPerChunk + (size_t)wave * DkvPartial<D>::kPerWave;
}

// Adds the chunks of every split key tile in chunk order (fixed order: the result does not
// depend on timing) and writes dK, dV. Bound by the partials' bytes (64 or 128 KB a chunk, from the memory-side
// cache), so the work is spread thin: a wavefront takes 32 keys x 32 columns of one tensor, four chunks
// of which it has in flight, and every workgroup finds the split tiles in the work list by itself (a few
// hundred entries). One workgroup per tile and KV head walked up to 32 chunks on a few dozen compute units:
// [1, 7424, 6/1 heads of 64] 52 -> 12 us, [1, 2432, 16/4 of 64] 25 -> 7, [4, 4096, 32/8 of 128] 22 -> 15,
// [2, 2432, 16/16 of 128] 19 -> 14, [4, 4224, 8/1 of 128] 25 -> 16.
// Where there are fewer such pieces than sets of four wavefronts, four wavefronts share one, 8 of its rows each,
// with 16 chunks in flight.
constexpr int kReduceGroups = 1024;
template <int WAVES>
struct DkvReduceLds {
  static constexpr int kMaxSplitTiles = kDkvSlots + 8;  // dkv_layout: at most half of max_partials <= 2 (kDkvSlots + 2)
  int2 split[kMaxSplitTiles];
  int wave_count[4][WAVES];
  __align__(16) bf16 patches[WAVES][32 * 32];
};
// Workgroup `group` of `groups`, WAVES wavefronts each (four or eight). Every backward call ends with a launch that does this, and
// it leaves the recomputing dQ kernel's work counters at zero, so that a later call on the same workspace can keep the work list and skip
// the kernel that builds it (and clears the counters). Nothing in such a launch uses them; an earlier pass of the call may have.
template <int D, int WAVES>
CT_DEVICE void dkv_reduce(const AttnParams& p, int group, int groups, DkvReduceLds<WAVES>& lds) {
  constexpr int kMaxSplitTiles = DkvReduceLds<WAVES>::kMaxSplitTiles;
  constexpr int kPieces = 2 * 4 * (D / 32);      // (tensor, wavefront of the dK/dV kernel, 32 columns)
  const int l = lane_id(), j = l & 31, half = l >> 5, w = uniform(threadIdx.x >> 6);
  const int nrb = p.S / 32;
  if (group == 0)
    for (int i = threadIdx.x; i < kDqCounters; i += 64 * WAVES) p.dq_counters[i] = 0;
  const int entries = uniform(p.dkv_header[0]);
  int tiles = 0;  // split tiles found, in list order (the same in every workgroup)
  for (int base = 0; base < entries; base += 256 * WAVES) {
    int2 entry[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int i = base + n * 64 * WAVES + threadIdx.x;
      entry[n] = i < entries ? p.dkv_entries[i] : make_int2(0, 0);
    }
    unsigned long long ballot[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      ballot[n] = __ballot((entry[n].y & 255) == 0 && ((entry[n].y >> 8) & 255) > 1);  // chunk 0 of several
      if (l == 0) lds.wave_count[n][w] = __popcll(ballot[n]);
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      if (base + n * 64 * WAVES >= entries) break;
      int at = tiles + __popcll(ballot[n] & ((1ull << l) - 1ull));
#pragma unroll
      for (int k = 0; k < WAVES; ++k) {
        if (k < w) at += lds.wave_count[n][k];
        tiles += lds.wave_count[n][k];
      }
      if ((ballot[n] >> l & 1) && at < kMaxSplitTiles) lds.split[at] = entry[n];
    }
    __syncthreads();
  }
  tiles = uniform(min(tiles, kMaxSplitTiles));
  const int items = tiles * p.Hkv * kPieces;
  const bool shared = items <= groups * (WAVES / 4);  // (then four wavefronts have one piece at most)
  const int set = w / 4, member = w % 4;
  for (int item = shared ? group * (WAVES / 4) + set : group * WAVES + w; item < items; item += groups * WAVES) {
    const int piece = item % kPieces, kvh = item / kPieces % p.Hkv;
    const int2 entry = lds.split[item / kPieces / p.Hkv];
    const int tile = uniform(entry.x), nsplit = uniform((entry.y >> 8) & 255), slot0 = uniform((unsigned)entry.y >> 16);
    const int db = piece % (D / 32), keys = piece / (D / 32) % 4, tensor = piece / (D / 32) / 4;
    const float* src = p.dkv_partials + dkv_partial_offset<D>(slot0, p.Hkv, kvh, keys) + tensor * DkvPartial<D>::kPerTensor +
                       db * 1024 + l * 4;
    const size_t chunk_stride = (size_t)p.Hkv * DkvPartial<D>::kPerChunk;
    const int b = tile / (nrb / 4), kt = tile % (nrb / 4);
    bf16* out = (tensor ? p.dv : p.dk) + (((size_t)b * p.S + (kt * 4 + keys) * 32) * p.Hkv + kvh) * D + db * 32;
    if (shared) {  // keys 8 member .. 8 member + 7 of the piece
      f32x4 sum = {};
      for (int c = 0; c < nsplit; c += 16) {
        f32x4 v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k)
          v[k] = c + k < nsplit ? *reinterpret_cast<const f32x4*>(src + (c + k) * chunk_stride + member * 256) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 16; ++k)
          if (c + k < nsplit) sum += v[k];
      }
      bf16* patch = lds.patches[w];
#pragma unroll
      for (int e = 0; e < 4; ++e) patch[(4 * half + e) * 32 + j] = (bf16)sum[e];
      __builtin_amdgcn_wave_barrier();
      const int row = l >> 2, chunk = (l & 3) * 8;
      if (row < 8)
        store_global16(out + (size_t)(8 * member + row) * p.Hkv * D + chunk, *reinterpret_cast<const u32x4*>(patch + row * 32 + chunk));
      return;
    }
    f32x4 sum[4] = {};
    for (int c = 0; c < nsplit; c += 4) {
      f32x4 v[4][4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[k][q] = c + k < nsplit ? *reinterpret_cast<const f32x4*>(src + (c + k) * chunk_stride + q * 256) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (c + k < nsplit)
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[q] += v[k][q];
    }
    // lane (j, half) holds column j of the keys 8 q + 4 half + e: through LDS to rows of 64 bytes
    bf16* patch = lds.patches[w];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) patch[(8 * q + 4 * half + e) * 32 + j] = (bf16)sum[q][e];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int row = (l >> 2) + 16 * n, chunk = (l & 3) * 8;
      store_global16(out + (size_t)row * p.Hkv * D + chunk, *reinterpret_cast<const u32x4*>(patch + row * 32 + chunk));
    }
  }
}

// On its own, the last kernel of a backward call.
template <int D>
__global__ __launch_bounds__(256) void attn_dkv_reduce_kernel(AttnParams p) {
  __shared__ DkvReduceLds<4> lds;
  dkv_reduce<D, 4>(p, blockIdx.x, gridDim.x, lds);
}

// Byte address of the dS block (key block rb with table entries ds_off / q_first, query block qb)
// of query head `head`, batch row b: wave-uniform.
CT_DEVICE char* ds_block_address(const AttnParams& p, int head, int b, int ds_off, int q_first, int qb) {
  const int first_head = p.kvh_base * (p.Hq / p.Hkv);
  const size_t block = ((size_t)(head - first_head) * p.B + b) * p.ds_row_blocks + (size_t)(ds_off + qb - q_first);
  return p.ds + block * kDsBlockBytes;
}

// A workgroup's place in the work list, by scalar loads that do not wait for one another.
struct DkvEntry {
  int tile, packed, entries;  // (how many the list has)
  CT_DEVICE explicit DkvEntry(const AttnParams& p) {
    const MetaPtr entry = meta_const(reinterpret_cast<const int*>(p.dkv_entries)) + 2 * (blockIdx.x / p.kvh_count);
    tile = entry[0];
    packed = entry[1];
    entries = meta_const(p.dkv_header)[0];
  }
};

// SPILL: every (key block, query block) step also stores its bf16 dS block to the dS region, for
// attn_dq_blocks_kernel.
//
// Head dimension 64 is held to 168 registers, three workgroups per compute unit (LDS has room for four): its steps are
// short and the vector ALU waits between the matrix instructions. With 177 registers and two workgroups:
// [2, 15616, 12/2 heads of 64] 544 -> 445 us, [1, 7424, 6/1] 95 -> 80. Its fragments are read ahead of the products
// (fragments_ahead): [1, 25472, 64/8], image blocks, 1800 -> 1690; the dQ kernel above likewise, 1280 -> 1190.
template <int D, bool SPILL>
CT_DEVICE void dkv_entry(const AttnParams& p, const lds_addr lds0, const DkvEntry& work) {
  if (SPILL && blockIdx.x == 0)  // work counters of the dQ kernel that reads the blocks
    for (int i = threadIdx.x; i < kDqCounters; i += 256) p.dq_counters[kDqCounters + i] = 0;
  constexpr int kStage = QdoStage<D>::kBytes;

  const int l = lane_id(), j = l & 31, half = l >> 5, w = uniform(threadIdx.x >> 6);
  const int nrb = p.S / 32;
  const int kvh = p.kvh_base + blockIdx.x % p.kvh_count, entry = blockIdx.x / p.kvh_count;
  // The way to the first products is a chain of memory round trips: the list's length and the entry (the grid is the list's
  // room, so it can be read whatever the length is), the tile's bounds beside its K and V rows, the first copies beside their
  // way into fragments. One after the other, and K and V by instructions that touch 32 rows each, the kernel took, us,
  // [3, 640, 12/2 heads of 128] 20.9 for 19.5, [4, 1792, 4/4] 26.7 for 25.2, [2, 2432, 16/16] 65.3 for 64.2, [4, 4096, 32/8],
  // documents of 64 to 300, 121.6 for 120.5, [8, 1152, 32/32 of 64], 16 to 64, 54.7 for 53.4.
  int tile = uniform(work.tile), packed = uniform(work.packed);
  asm volatile("" : "+s"(tile), "+s"(packed));
  if (entry >= uniform(work.entries) || (D == 128 && !SPILL && other_dkv_kernel(p, false))) return;
  const int chunk = packed & 255, nsplit = (packed >> 8) & 255, slot0 = (unsigned)packed >> 16;
  const int b = tile / (nrb / 4), kt = tile % (nrb / 4);
  const int g = p.Hq / p.Hkv;
  const int* meta_b = p.meta + (size_t)b * nrb * kMetaW;
  const RowFragOffsets<D / 8> ro(lds0);
  const TrFragOffsets<D / 8, KSlots::kAccum> to(lds0);

  const int my_rb = kt * 4 + w;
  const int key = my_rb * 32 + j;
  const int seg_k = p.seg[(size_t)b * p.S + key];
  const bool has_end = p.end != nullptr;
  const size_t kv_row_stride = (size_t)p.Hkv * D;
  const size_t kv_off = (((size_t)b * p.S + my_rb * 32) * p.Hkv + kvh) * D;
  // (V at D = 64 directly, for the addresses at which it is stored: they stay for the loop's reads. Without them the compiler
  // forms them in every step, and the kernel is 4 % slower with long documents.)
  RowBlockLoader<D> k_rows, v_rows;
  k_rows.request(p.k + kv_off, kv_row_stride);
  if constexpr (D == 128) {
    v_rows.request(p.v + kv_off, kv_row_stride);
  } else {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) v_rows.raw[ks] = load_global16(p.v + kv_off + j * kv_row_stride + 16 * ks + 8 * half);
  }

  int q_lo = INT_MAX, q_hi = -1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const MetaPtr m = meta_const(meta_b + (kt * 4 + i) * kMetaW);
    q_lo = min(q_lo, uniform(m[kQFirst]));
    q_hi = max(q_hi, uniform(m[kQLast]));
  }
  // (the extremes of several come out of the vector unit, and what is selected and added by them would stay there)
  q_lo = uniform(q_lo);
  q_hi = uniform(q_hi);
  const int my_min = uniform(meta_const(meta_b)[my_rb * kMetaW + kMinNz]);
  const int my_max = uniform(meta_const(meta_b)[my_rb * kMetaW + kMaxId]);
  const int my_uni = uniform(meta_const(meta_b)[my_rb * kMetaW + kUniform]);
  const int my_q_first = uniform(meta_const(meta_b)[my_rb * kMetaW + kQFirst]);
  const int my_ds_off = uniform(meta_const(meta_b)[my_rb * kMetaW + kDsOff]);

  // K fragments stay in registers; V fragments are parked in LDS (this wavefront's
  // private 32-row patch) and re-read per block, which keeps the kernel under 256
  // registers so that two workgroups share a CU.
  const int vpatch_off = QdoStage<D>::kVResident + w * 32 * D * 2;
  const lds_addr vpatch = lds0 + vpatch_off;
  f32x16 dkacc[D / 32], dvacc[D / 32];  // (D = 128: in accumulation registers until the end)
  if constexpr (D == 128) {
    asm volatile(CT_DKV_ZERO : : : CT_DKV_ACCUMULATORS);
  } else {
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      dkacc[db] = zero16();
      dvacc[db] = zero16();
    }
  }

  // The Q tiles stay unscaled in LDS: the softmax scale enters the exponent in f32
  // (S = scale * (Q K^T); the forward rounded scale * Q to bf16 first, a difference of one
  // bf16 rounding per element of Q) and dK = scale * (dS^T Q) is scaled once at the end.
  const float scale_log2e = exponent_scale(p.scale) * kLog2e;
  const float masked = masked_score(p.scale);

  // Work items: (head of the group, query block) pairs, flattened; query block fastest.
  const int nq = (q_lo <= q_hi) ? (q_hi - q_lo + 1) : 0;
  const int per_chunk = (nq * g + nsplit - 1) / nsplit;
  int it = chunk * per_chunk;
  const int items = min(nq * g, it + per_chunk);  // end of this chunk's item range
  const TileDma<kQueryTile, D / 8> dma((size_t)p.Hq * D * 2);
  // (a chunk without items: an address inside the arrays all the same)
  QdoCursor<D> next(p, b, uniform(kvh * g + (it < items ? it / nq : 0)), uniform(it < items ? q_lo + it % nq : 0), q_lo, q_hi, w);
  if (it < items) next.fetch(dma, lds0, w);
  // Make the K fragment loads complete here. Left pending, their first use inside the item
  // loop gets an `s_waitcnt vmcnt(n)` whose count fits the first item only; on every later item
  // the same wait stalls until the asynchronous copies of the next stage have landed.
  bf16x8 kf[D / 16];
  k_rows.to_fragments(vpatch, kf);
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) asm volatile("" : "+v"(kf[ks]));
  if constexpr (D == 128) {
    v_rows.to_patch(vpatch);
  } else {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) lds_store<u32x4>(ro.addr(vpatch_off, 0, ks), v_rows.raw[ks]);
  }
  dma_wait_all();
  __syncthreads();

  QueryBlockBounds qb_bounds = next.query_bounds();
  auto step = [&](auto stage_tag) {
    constexpr int CUR = decltype(stage_tag)::value;
    const lds_addr stage = lds0 + CUR * kStage;
    const int qb = q_hi - next.left, head = next.head;
    // bounds of this query block, read one item ahead
    const int q_min = qb_bounds.min_nz, q_max = qb_bounds.max_id, q_end_max = qb_bounds.end_max,
              q_end_min = qb_bounds.end_min, q_uni = qb_bounds.uniform;
    if (it + 1 < items) {
      next.advance(nq);
      next.fetch(dma, lds0 + (CUR ^ 1) * kStage, w);
    }
    QueryBlockBounds bounds_ahead;  // (behind the last item: the same bounds again)
    const bool visit = blocks_interact(q_min, q_max, q_end_max, my_min, my_max, my_rb * 32);
    if (D != 64 || !visit) bounds_ahead = next.query_bounds();
    if (!visit) {
    } else if constexpr (D == 128) {
      const bool interior = tile_is_interior(q_uni, q_end_min, my_uni, my_rb * 32 + 31);
      const int seg_k_or_never = seg_k != 0 ? seg_k : -1;  // ids are >= 0
      char* block = SPILL ? ds_block_address(p, head, b, my_ds_off, my_q_first, qb) : nullptr;
      const unsigned lane16 = SPILL ? (unsigned)lane_id_here() * 16 : 0;
      const DkvFrame f{ro, to, kf, lds0 + 16 * half, scale_log2e, (unsigned)vpatch_off};
      if (interior)
        dkv_step_128<CUR * kStage, DkvPairs::kAll, SPILL>(f, masked, 0, 0, block, lane16);
      else if (has_end)
        dkv_step_128<CUR * kStage, DkvPairs::kToEnds, SPILL>(f, masked, seg_k_or_never, key, block, lane16);
      else
        dkv_step_128<CUR * kStage, DkvPairs::kToRows, SPILL>(f, masked, seg_k_or_never, key - 4 * half - qb * kQueryTile, block,
                                                             lane16);
    } else {
      // The row offsets below depend on the lane only; hoisted out of the loop they become
      // spilled registers whose reloads wait for every copy in flight. Recompute them here.
      int half_here = half;
      asm volatile("" : "+v"(half_here));
      // Both products start from the per-row terms of their 16 query rows instead of zero (the
      // statistics pass left -lse / scale and -delta): the sums S - lse / scale and dP - delta
      // come out of the matrix pipe, and no vector instruction adds them.
      f32x16 s, dp;
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int r0 = 8 * qd + 4 * half_here;
        const f32x4 lse4 = lds_load<f32x4>(stage + QdoStage<D>::kLse + r0 * 4);
        const f32x4 del4 = lds_load<f32x4>(stage + QdoStage<D>::kDelta + r0 * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[4 * qd + e] = lse4[e];
          dp[4 * qd + e] = del4[e];
        }
      }
      constexpr int kSteps = D / 16, qOff = CUR * kStage + QdoStage<D>::kQ, doOff = CUR * kStage + QdoStage<D>::kDo;
      fragments_ahead<kSteps, kSteps>([&](int i) { return ro.load(qOff, 0, i); },
                                      [&](int i, bf16x8 queries) { s = mfma32(queries, kf[i], s); });
      struct Pair {
        bf16x8 dout, v;
      };
      fragments_ahead<kSteps, 2>([&](int i) { return Pair{ro.load(doOff, 0, i), ro.load(vpatch_off, 0, i)}; },
                                 [&](int i, const Pair& rows) { dp = mfma32(rows.dout, rows.v, dp); });
      bounds_ahead = next.query_bounds();  // (a wait for LDS reads is one for all scalar loads too)
      const bool interior = tile_is_interior(q_uni, q_end_min, my_uni, my_rb * 32 + 31);
      f32x16 prob;
      if (!interior) {
        // Masked scores become -inf (their probability is then exactly 0). Written with
        // bitwise logic and selects only: the per-element tests must not turn into branches.
        const int seg_k_or_never = seg_k != 0 ? seg_k : -1;  // ids are >= 0
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const int r0 = 8 * qd + 4 * half_here;  // first of 4 consecutive query rows
          const i32x4 seg4 = lds_load<i32x4>(stage + QdoStage<D>::kSeg + r0 * 4);
          i32x4 end4;
          if (has_end) {
            end4 = lds_load<i32x4>(stage + QdoStage<D>::kEnd + r0 * 4);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) end4[e] = qb * kQueryTile + r0 + e;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool ok = (seg4[e] == seg_k_or_never) & (key <= end4[e]);
            s[4 * qd + e] = ok ? s[4 * qd + e] : masked;
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pr = exp2_fast(s[r] * scale_log2e);  // s = S - lse / scale
        prob[r] = pr;
        dp[r] = pr * dp[r];                              // dp = dP - delta
      }
      if constexpr (SPILL) {
        // The block as the lanes hold it: the two operands of the dK product (8 query rows of one
        // key each) as two runs of 64 x 16 bytes in lane order, so a store writes 1 KB end to end.
        char* block = ds_block_address(p, head, b, my_ds_off, my_q_first, qb);
        const unsigned lane_off = (unsigned)lane_id_here() * 16;
        store_global16_s<0>(block, lane_off, __builtin_bit_cast(f32x4, pack_acc8(dp, 0)));
        store_global16_s<1024>(block, lane_off, __builtin_bit_cast(f32x4, pack_acc8(dp, 1)));
      }
      const bf16x8 keys[4] = {pack_acc8(prob, 0), pack_acc8(prob, 1), pack_acc8(dp, 0), pack_acc8(dp, 1)};
      constexpr int kBlocks = D / 32;
      fragments_ahead<4 * kBlocks, 4>(
          [&](int i) {
            return to.load(CUR * kStage + (i < 2 * kBlocks ? QdoStage<D>::kDo : QdoStage<D>::kQ), i / kBlocks % 2, i % kBlocks);
          },
          [&](int i, bf16x8 rows) {
            f32x16& acc = (i < 2 * kBlocks ? dvacc : dkacc)[i % kBlocks];
            acc = mfma32(keys[i / kBlocks], rows, acc);
          });
    }
    // The next block's bounds are waited for here, where the step has given them the time. Left to their first use
    // the wait stands in the next step behind the loads for the step after it, and as scalar loads return in any
    // order it waits for those too: a round trip of the scalar cache in every step.
    bounds_ahead.pin();
    qb_bounds = bounds_ahead;
    // Vector memory operations complete in the order they were issued: the two stores of this
    // step are the youngest, so waiting for all but two has waited for every copy of the next
    // stage without waiting for the stores (they are long done one step later).
    if (SPILL && visit) __builtin_amdgcn_s_waitcnt(0x0F72);
    else dma_wait_all();
    __syncthreads();
    ++it;
  };
  while (it < items) {
    step(std::integral_constant<int, 0>{});
    if (it >= items) break;
    step(std::integral_constant<int, 1>{});
  }

  if constexpr (D == 128) {
    // The last sums have left the matrix pipe after these wait states (the compiler does not see the MFMAs).
    asm volatile("s_nop 15\n\ts_nop 7" : : : "memory");
    float* mine = nsplit > 1 ? p.dkv_partials + dkv_partial_offset<D>(slot0 + chunk, p.Hkv, kvh, w) : nullptr;
    const size_t out_off = (((size_t)b * p.S + my_rb * 32) * p.Hkv + kvh) * D;
    leave_accumulators<4, true>(p.scale, mine, vpatch, p.dk + out_off, kv_row_stride);
    leave_accumulators<0, false>(p.scale, mine ? mine + DkvPartial<D>::kPerTensor : nullptr, vpatch, p.dv + out_off, kv_row_stride);
    return;
  }
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) dkacc[db][e] *= p.scale;

  if (nsplit > 1) {
    // A chunk of a split tile leaves its sums as f32 for attn_dkv_reduce_kernel:
    // [dK | dV][wavefront][d block][register quad][lane][4], 16 bytes per lane and store.
    float* mine = p.dkv_partials + dkv_partial_offset<D>(slot0 + chunk, p.Hkv, kvh, w) + l * 4;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        f32x4 a, c;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[e] = dkacc[db][4 * q4 + e];
          c[e] = dvacc[db][4 * q4 + e];
        }
        *reinterpret_cast<f32x4*>(mine + (db * 4 + q4) * 256) = a;
        *reinterpret_cast<f32x4*>(mine + DkvPartial<D>::kPerTensor + (db * 4 + q4) * 256) = c;
      }
    return;
  }

  const lds_addr patch = vpatch;  // V fragments are no longer needed
  const size_t out_off = (((size_t)b * p.S + my_rb * 32) * p.Hkv + kvh) * D;
  store_rows<D>(dkacc, patch, p.dk + out_off, kv_row_stride);
  __builtin_amdgcn_wave_barrier();
  store_rows<D>(dvacc, patch, p.dv + out_off, kv_row_stride);
}

template <int D, bool SPILL>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_dkv_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  dkv_entry<D, SPILL>(p, lds_address_of(smem_raw), DkvEntry(p));
}

// With the stores or without them, as the header says. (Two kernels, one of them to exit at once, would be one more launch; with
// both bodies in one a few scalar registers and 12 bytes of scratch a lane go to what the loops do not use.)
template <int D>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_dkv_choice_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  const DkvEntry entry(p);
  if (dq_recomputes(p)) dkv_entry<D, false>(p, lds_address_of(smem_raw), entry);
  else dkv_entry<D, true>(p, lds_address_of(smem_raw), entry);
}

// The same for launches in which the recomputing dQ has none of its own: where the header asks for it the workgroups, as many as
// the list has room, go on with query tiles when they have left their key tile, and the tiles fill what the list leaves at its
// end. (Workgroups of their own behind the list's: 768 more to start for nothing, 1 us of 19 with short documents. The answer read
// by a vector load, a round trip in front of the entry's: 0.98 of the time then; three scalar loads side by side: 0.997.)
// Backward kernels, us, stored blocks / so: [1, 4096, 24/8 heads of 64], documents of 2048 to 4096 225 / 188, whole rows 263 / 212;
// [3, 2048, 32/8] whole rows 272 / 212, of 16 to 64 72.0 / 71.9; [1, 3456, 48/8], images, 385 / 278; [7, 1024, 32/32], of 512 to 1024
// 136 / 119, of 100 to 200 88.9 / 89.4.
template <int HS>
__global__ __launch_bounds__(256, 3) void attn_dkv_then_dq_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  __shared__ int next_pull;
  const lds_addr lds0 = lds_address_of(smem_raw);
  const DkvEntry entry(p);
  if (!dq_recomputes(p)) {
    dkv_entry<64, true>(p, lds0, entry);
    return;
  }
  dkv_entry<64, false>(p, lds0, entry);
  __syncthreads();  // the store patches become stages
  attn_dq_tiles<64, HS, 3, false>(p, blockIdx.x, gridDim.x, lds0, &next_pull);
}

// ---------------------------------------------------------------------------
// dQ from stored dS blocks: dQ = scale * sum over visited key blocks of dS K
// (src/kernels/efficient_attention.py:1046-1048 with the dS of :1040-1045 read back instead of
// formed again). Same workgroup shape, work pulling and key-tile walk as attn_dq_kernel; a stage
// holds the K rows of a 64-key tile (shared by the 4 wavefronts) and, per wavefront, the dS blocks
// of its query block against the tile's two key blocks, copied straight from the dS region. A
// block is read back as the B operand of dQ^T += K^T dS^T with transposing LDS reads, which is
// the transposition between the key-stationary kernel that wrote it (lanes along keys) and this
// query-stationary product (lanes along queries). Bound by the bytes of the blocks it reads.
// ---------------------------------------------------------------------------
// Eight wavefronts per workgroup (HS heads x 8 / HS query blocks). A stage: the K rows of one
// 32-key block (shared by all wavefronts) and, per wavefront, the dS block of its query block
// against that key block. A dS block sits in LDS as it sits in memory (two runs of 64 x 16 bytes,
// lane (half, key) order), the second run 64 bytes further than its 1 KB so that the transposing
// reads of one fragment spread over all banks. Three stages: two key blocks are in flight while
// one is worked on (the kernel lives on bytes in flight; what bounds them is LDS, and with eight
// wavefronts per K block four fifths of a stage are dS).
//
// KS > 1: KS wavefronts share the key blocks of a row block, every KS-th block each (a stage holds the K rows of
// KS blocks), and add their sums through LDS in a fixed order at the end: for launches of few row blocks, whose
// time is the walk of the longest row.
constexpr int kDqbWaves = 8;
template <int D, int KS>
struct DsStage {
  static constexpr int kK = 0;
  static constexpr int kKBytes = 32 * D * 2;  // of one key block
  static constexpr int kRun = 1024 + 64;
  static constexpr int kPatch = 2 * kRun;
  static constexpr int kDs = KS * kKBytes;  // [wavefront][kPatch]
  static constexpr int kBytes = kDs + kDqbWaves * kPatch;
  static constexpr int kStages = 3;
  static constexpr int kMergeBytes = 64 * (D / 2) * 4;  // the sums that a wavefront hands over
  static constexpr int kStorePatches = (kDqbWaves - kDqbWaves / KS) * kMergeBytes;
  static constexpr int kEndBytes = kStorePatches + kDqbWaves / KS * 32 * D * 2;
  static constexpr int kTotalBytes = kStages * kBytes > kEndBytes ? kStages * kBytes : kEndBytes;
  // the workgroup's copies of a stage's K rows: by all threads, or by half of them for a small block
  static constexpr int kCopyThreads = KS * kKBytes >= 8192 ? 512 : 256;
  typedef TileDma<KS * 32, D / 8, kCopyThreads> KDma;
};

// Transposed-fragment pointers into a dS block: the B operand of dQ^T += K^T dS^T wants, for
// query slot n = lane % 32, the keys of a k-step in accumulator order (matching the K fragments).
// The 8-byte piece (key, slots 4 m .. 4 m + 3) is the half (slots & 4) of lane (half = slot >> 4,
// key)'s 16 bytes in run (slot >> 3) & 1.
struct DsFragPtrs {
  lds_addr ptr[2];
  CT_DEVICE DsFragPtrs(lds_addr base, int l) {
    const int pp = l & 15, q16 = (l >> 4) & 1, half = l >> 5;
#pragma unroll
    for (int second = 0; second < 2; ++second) {
      const int key = 4 * half + 8 * second + (pp >> 2);
      const int run = (pp & 3) >> 1, piece = pp & 1;
      ptr[second] = base + (run * (1024 + 64) + q16 * 512 + key * 16 + piece * 8);
    }
  }
  // keys 16 ks .. 16 ks + 15 of the block at byte offset `off`
  CT_DEVICE bf16x8 load(int off, int ks) const {
    const bf16x4_vs lo = lds_load_tr(ptr[0] + (off + ks * 256));
    const bf16x4_vs hi = lds_load_tr(ptr[1] + (off + ks * 256));
    bf16x8 out;
    out[0] = lo[0]; out[1] = lo[1]; out[2] = lo[2]; out[3] = lo[3];
    out[4] = hi[0]; out[5] = hi[1]; out[6] = hi[2]; out[7] = hi[3];
    return out;
  }
};

// What the walk needs to know about a 32-key block (scalar loads).
struct DsKeyBlockInfo {
  int k_min, k_max, q_first, ds_off;
};
CT_DEVICE DsKeyBlockInfo ds_key_block_info(const int* meta_b, int rbk) {
  const MetaPtr m = meta_const(meta_b + rbk * kMetaW);
  DsKeyBlockInfo info;
  info.k_min = m[kMinNz];
  info.k_max = m[kMaxId];
  info.q_first = m[kQFirst];
  info.ds_off = m[kDsOff];
  return info;
}

// store_rows_t for an accumulator whose lane j holds the query row ds_slot_row(j) of the block.
template <int D>
CT_DEVICE void store_slot_rows_t(const f32x16* acc, float row_scale, lds_addr patch, bf16* gbase,
                                 size_t row_stride) {
  constexpr int CPR = D / 8;
  int l = lane_id();
  asm volatile("" : "+v"(l));
  const int row_of_lane = ds_slot_row(l & 31), half = l >> 5;
  using Patch = PatchRows<D>;
  const lds_addr store_base = Patch::store_base(patch, row_of_lane, half);
  const unsigned row_swizzle = Patch::row_swizzle(row_of_lane);
  auto block = [&](auto db_tag) {
    constexpr int db = decltype(db_tag)::value;
    auto quad = [&](auto qd_tag) {
      constexpr int qd = decltype(qd_tag)::value;
      bf16x4 pk;
#pragma unroll
      for (int e = 0; e < 4; ++e) pk[e] = (bf16)(acc[db][4 * qd + e] * row_scale);
      lds_store<bf16x4>(store_base + Patch::template chunk_term<db * 4 + qd>(row_swizzle), pk);
    };
    quad(std::integral_constant<int, 0>{});
    quad(std::integral_constant<int, 1>{});
    quad(std::integral_constant<int, 2>{});
    quad(std::integral_constant<int, 3>{});
  };
  block(std::integral_constant<int, 0>{});
  block(std::integral_constant<int, 1>{});
  if constexpr (D > 64) {
    block(std::integral_constant<int, 2>{});
    block(std::integral_constant<int, 3>{});
  }
  static_assert(D == 64 || D == 128, "two or four 32-column blocks");
  (void)CPR;
  __builtin_amdgcn_wave_barrier();
  Patch::to_global(patch, l, gbase, row_stride);
}

// s_waitcnt vmcnt(n) for a wave-uniform n that is one of the few values the walk produces.
template <int MOST>
CT_DEVICE void wait_all_copies_but(int n) {
  if constexpr (MOST == 0) __builtin_amdgcn_s_waitcnt(0x0F70);
  else if (n >= MOST) __builtin_amdgcn_s_waitcnt(0x0F70 | MOST);
  else wait_all_copies_but<MOST - 1>(n);
}

template <int D, int HS, int KS>
CT_DEVICE void attn_dq_blocks_item(const AttnParams& p, int b, int kvh, int slice, int qt, const lds_addr lds0,
                                   const typename DsStage<D, KS>::KDma& kdma, const DsFragPtrs& frags,
                                   const TrFragOffsets<D / 8, KSlots::kAccum>& tp) {
  using Stage = DsStage<D, KS>;
  constexpr int kSlots = kDqbWaves / KS, PB = kSlots / HS;
  constexpr int kStage = Stage::kBytes, kMostCopies = Stage::KDma::kPasses + 2;
  const int nrb = p.S / 32;
  const int g = p.Hq / p.Hkv;
  const int w = uniform(threadIdx.x >> 6), slot = w % kSlots, share = w / kSlots;
  const int h = kvh * g + slice * HS + (slot % HS);
  int rb = qt * PB + (slot / HS);
  const bool active = rb < nrb;
  if (!active) rb = nrb - 1;
  const int* meta_b = p.meta + (size_t)b * nrb * kMetaW;
  QueryBlockBounds mine = query_block_bounds(meta_b, rb);
  if (!active) mine.min_nz = 0;  // interacts with nothing
  int first_tile = INT_MAX, last_tile = -1;  // 64-key tiles, as the table has them
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    if (qt * PB + i >= nrb) break;
    const MetaPtr m = meta_const(meta_b + (qt * PB + i) * kMetaW);
    first_tile = min(first_tile, uniform(m[kKvFirst]));
    last_tile = max(last_tile, uniform(m[kKvLast]));
  }
  // the walk is in steps of KS 32-key blocks (a tile without keys is the pair INT_MAX / -1: converted only
  // when there is a range, and clamped to the row so that no table entry can lead outside it; rows are whole
  // numbers of 4 blocks)
  const bool any = first_tile <= last_tile && first_tile >= 0 && last_tile < nrb / 2;
  const int first = any ? 2 * first_tile / KS : 0;
  const int last = any ? (2 * last_tile + 1) / KS : -1;
  const char* kbase = reinterpret_cast<const char*>(p.k + ((size_t)b * p.S * p.Hkv + kvh) * D);
  const size_t kv_row_bytes = (size_t)p.Hkv * D * 2;
  const unsigned ds_lane_off = (unsigned)lane_id_here() * 16;
  const int my_ds = Stage::kDs + w * Stage::kPatch;  // this wavefront's block inside a stage
  const bool copies_k = w < Stage::kCopyThreads / 64;

  f32x16 dqacc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db) dqacc[db] = zero16();

  const auto info_of = [&](int t) { return ds_key_block_info(meta_b, t * KS + share); };  // this wavefront's block of step t
  auto visits = [&](const DsKeyBlockInfo& info, int t) {
    return blocks_interact(mine.min_nz, mine.max_id, mine.end_max, uniform(info.k_min), uniform(info.k_max),
                           (t * KS + share) * 32);
  };
  // K rows of step t (all wavefronts) and this wavefront's dS block against its share; returns the
  // number of copy instructions this wavefront issued
  auto issue = [&](int t, const DsKeyBlockInfo& info, lds_addr stage) {
    int issued = 0;
    if (copies_k) {
      kdma.issue(kbase + (size_t)t * (KS * 32) * kv_row_bytes, stage + Stage::kK);
      issued = Stage::KDma::kPasses;
    }
    if (visits(info, t)) {
      const char* block = ds_block_address(p, h, b, uniform(info.ds_off), uniform(info.q_first), rb);
      dma16_s(block, ds_lane_off, stage + my_ds);
      dma16_s(block + 1024, ds_lane_off, stage + (my_ds + Stage::kRun));
      issued += 2;
    }
    return issued;
  };

  // cur, next, after: steps t, t + 1, t + 2; the stage of step t + i is (stage of t + i) mod 3
  int t = first;
  DsKeyBlockInfo cur = {}, next = {}, after = {};
  int pending = 0;  // copy instructions of the youngest step in flight
  if (t <= last) {
    cur = info_of(t);
    issue(t, cur, lds0);
    if (t + 1 <= last) {
      next = info_of(t + 1);
      pending = issue(t + 1, next, lds0 + kStage);
      if (t + 2 <= last) after = info_of(t + 2);
    }
  }
  wait_all_copies_but<kMostCopies>(pending);
  __syncthreads();

  auto step = [&](auto stage_tag) {
    constexpr int CUR = decltype(stage_tag)::value;
    constexpr int kFill = (CUR + 2) % 3;  // last read one step ago: every wavefront is past that barrier
    DsKeyBlockInfo later = after;
    pending = 0;
    if (t + 2 <= last) {
      pending = issue(t + 2, after, lds0 + kFill * kStage);
      if (t + 3 <= last) later = info_of(t + 3);
    }
    if (visits(cur, t)) {
      constexpr int ds_off = CUR * kStage;  // + my_ds, inside the pointers
      constexpr int k_off = CUR * kStage + Stage::kK;  // + this wavefront's share, inside the pointers
      const bf16x8 ds0 = frags.load(ds_off, 0), ds1 = frags.load(ds_off, 1);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) dqacc[db] = mfma32(tp.load(k_off, 0, db), ds0, dqacc[db]);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) dqacc[db] = mfma32(tp.load(k_off, 1, db), ds1, dqacc[db]);
    }
    // Copies complete in the order they were issued: all but the ones just issued means step t + 1
    // has landed.
    wait_all_copies_but<kMostCopies>(pending);
    __syncthreads();
    cur = next;
    next = after;
    after = later;
    ++t;
  };
  while (t <= last) {
    step(std::integral_constant<int, 0>{});
    if (t > last) break;
    step(std::integral_constant<int, 1>{});
    if (t > last) break;
    step(std::integral_constant<int, 2>{});
  }

  if constexpr (KS > 1) {
    // (the walk's last barrier is behind every read of the stages)
    if (share > 0) {
      const lds_addr sums = lds0 + (w - kSlots) * Stage::kMergeBytes + lane_id_here() * 16;
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          lds_store<f32x4>(sums + (db * 4 + qd) * 1024,
                           f32x4{dqacc[db][4 * qd], dqacc[db][4 * qd + 1], dqacc[db][4 * qd + 2], dqacc[db][4 * qd + 3]});
    }
    __syncthreads();
    if (share > 0) return;
#pragma unroll
    for (int other = 1; other < KS; ++other) {
      const lds_addr sums = lds0 + ((other - 1) * kSlots + slot) * Stage::kMergeBytes + lane_id_here() * 16;
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const f32x4 o = lds_load<f32x4>(sums + (db * 4 + qd) * 1024);
#pragma unroll
          for (int e = 0; e < 4; ++e) dqacc[db][4 * qd + e] += o[e];
        }
    }
  }
  if (active) {
    const lds_addr patch = lds0 + (Stage::kStorePatches + slot * (32 * D * 2));
    bf16* gbase = p.dq + (((size_t)b * p.S + rb * 32) * p.Hq + h) * D;
    store_slot_rows_t<D>(dqacc, p.scale, patch, gbase, (size_t)p.Hq * D);
  }
  if constexpr (KS == 1) {
    // the store patches overlap the stages of the next item
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __syncthreads();
  }
}

// The last reduce_groups workgroups add the chunks of split key tiles (dkv_reduce). The two passes read what the dK/dV kernel
// left and write different tensors; the sums are few bytes a place and take the places that tiles leave free: where a workgroup
// has one tile (KS > 1) beside them, where the workgroups pull tiles (KS = 1) when the first of those end. Both in launches of
// their own / in this one, us: [4, 4096, 32/8 heads of 128], documents of 64 to 4096, 203 + 15 / 206, [2, 10496, 12/4], 248 to
// 3277, 81 + 18 / 86, [4, 4096, 8/1] 90 + 19 / 93, [2, 8192, 16/16], 64 to 2000, 100 + 5 / 100. The sums clear the recomputing
// kernel's work counters, so this kernel has counters of its own.
template <int D, int HS, int KS>
__global__ __launch_bounds__(kDqbWaves * 64, 2) void attn_dq_blocks_kernel(AttnParams p, int reduce_groups) {
  extern __shared__ __align__(16) char smem_raw[];
  {
    typedef DkvReduceLds<kDqbWaves> ReduceLds;
    static_assert(sizeof(ReduceLds) <= DsStage<D, KS>::kTotalBytes, "the sums' list and patches fit");
    const int group = (int)blockIdx.x - ((int)gridDim.x - reduce_groups);
    if (group >= 0) {
      dkv_reduce<D, kDqbWaves>(p, group, reduce_groups, *reinterpret_cast<ReduceLds*>(smem_raw));
      return;
    }
  }
  // (beside the first reads of the schedule for a workgroup per tile, whose time this round trip would be part of)
  const int recomputes = D == 64 && p.ds_most_blocks ? meta_const(p.dkv_header)[kDqRecomputes] : 0;
  if (KS == 1 && uniform(recomputes) != 0) return;
  const lds_addr lds0 = lds_address_of(smem_raw);
  __shared__ int next_pull;
  using Stage = DsStage<D, KS>;
  constexpr int PB = kDqbWaves / KS / HS;
  const int nrb = p.S / 32;
  const int slices = (p.Hq / p.Hkv) / HS;
  const int groups = slices * p.kvh_count;
  const int group = blockIdx.x % groups, member = blockIdx.x / groups, members = (gridDim.x - reduce_groups) / groups;
  const int kvh = p.kvh_base + group % p.kvh_count, slice = group / p.kvh_count;
  const int tpr = bin_tiles_per_row(nrb, PB);
  const int total = p.B * tpr;
  const MetaPtr sched = meta_const(p.sched + query_schedule_offset(nrb, PB));
  const bool dynamic = slices * p.Hkv <= kDqCounters;
  int* counters = p.dq_counters + kDqCounters;
  const typename Stage::KDma kdma((size_t)p.Hkv * D * 2);
  const int w = threadIdx.x >> 6;
  const DsFragPtrs frags(lds0 + (Stage::kDs + w * Stage::kPatch), lane_id());
  const TrFragOffsets<D / 8, KSlots::kAccum> tp(lds0 + w / (kDqbWaves / KS) * Stage::kKBytes);
  if constexpr (KS > 1) {  // a workgroup per tile, heaviest first
    const int b = member % p.B, tile = sched[(size_t)b * schedule_ints(nrb) + member / p.B];
    if (uniform(recomputes) != 0) return;
    const int qt = uniform(tile);
    attn_dq_blocks_item<D, HS, KS>(p, b, kvh, slice, qt, lds0, kdma, frags, tp);
    return;
  }
  for (int pull = member;; pull += members) {
    if (dynamic) {
      if (threadIdx.x == 0) next_pull = atomicAdd(&counters[slice * p.Hkv + kvh], 1);
      __syncthreads();
      pull = uniform(next_pull);
      __syncthreads();
    }
    if (pull >= total) break;
    const int b = pull % p.B, rank = pull / p.B;
    const int qt = uniform(sched[(size_t)b * schedule_ints(nrb) + rank]);
    if constexpr (KS == 1) attn_dq_blocks_item<D, HS, KS>(p, b, kvh, slice, qt, lds0, kdma, frags, tp);
  }
}

}  // namespace ct
