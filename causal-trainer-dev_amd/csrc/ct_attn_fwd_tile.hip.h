// Attention forward at head dimension 128: the interleaved statements of attn_fwd_item (ct_attn_kernels.hip.h) in workgroups of
// four wavefronts, two per compute unit, one query tile each, dealt by the hardware heaviest first.
//
// The workgroup of eight that walks work bins has all wavefronts of a compute unit in one phase: what a query tile spends before
// its first scores and behind its last ones (15 of 40 thousand clocks at (4, 4096, 32/8), documents of 64 to 4096) nobody uses.
// Here the other workgroup does, the launch ends evenly whatever the documents are, and row blocks of padding cost a store.
// The price is that a staged key tile serves 128 instead of 256 rows; two things pay for it:
//
//   * all eight copies of a step ride behind the MFMAs of its first statement (issued in front of it: 3 to 5 % of whole rows);
//   * inside a stretch of tiles seen in full a step takes no maximum and no decision (free_step): the exponentials, 3.5 vector
//     instructions per MFMA for 4.3, are formed against the reference as it is, behind all 32 MFMAs. Floats scale: a row sum may
//     grow to 2^30 against an old reference with nothing lost. From there on the tile's steps follow the maximum again; should
//     a sum pass 2^60 or be no number, the workgroup runs its tile once more with the maximum in every step.
//
// Measured, us, workgroups of eight / this: (4, 4096, 32/8) documents of 64 to 4096 197 / 190, whole rows 492 / 483;
// (2, 8192, 16/16) images 191 / 180; (1, 32768, 64/8) documents of 512 to 32768 6700 / 6600; (2, 2560, 48/16) of 176 to 2492
// 78.7 / 65; (4, 2432, 48/8) images 193 / 172; (3, 2432, 64/16) of 53 to 204 95 / 80; (1, 3840, 64/16) images 71 / 58;
// 240 shapes of 2048 row blocks and more 1.07 in the geometric mean. Not better: see dispatch_fwd.
#pragma once

#include "ct_attn_kernels.hip.h"

namespace ct {

constexpr int kTileWaves = 4;
// A lane's row sum from which on a tile's steps follow the maximum again, and from which on the tile is run again.
constexpr float kFollowFromSum = 0x1p30f, kLostFromSum = 0x1p60f;
// Workgroups from which on the tiles of a batch row go out sixteen at a time (attn_fwd_tile_kernel).
constexpr unsigned kRowsInTurnFrom = 3072;

// LDS: stages as VkStage, the ring of key ids, and a word that says whether the tile has to be run again. The second stage is
// also where the Q rows pass through, and both are store patches in the end.
struct FwdTileStage {
  static constexpr int kV = 0, kK = kKeyTile * 256, kBytes = 2 * kKeyTile * 256;
  static constexpr int kSegRing = 2 * kBytes, kSegSlotBytes = kKeyTile * 4;
  static constexpr int kLost = kSegRing + 4 * kSegSlotBytes;
  static constexpr int kTotalBytes = kLost + 16;
  static constexpr int kPatchBytes = 32 * 256;  // of a wavefront
  static_assert(kTileWaves * kPatchBytes <= kBytes, "the patches fit in a stage");
  static_assert(2 * kTotalBytes <= 160 * 1024, "two workgroups per compute unit");
  static CT_DEVICE int seg_slot(int t) { return kSegRing + (t & 3) * kSegSlotBytes; }
};

template <int HS>
__global__ __launch_bounds__(kTileWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_fwd_tile_kernel(AttnParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  using Stage = FwdTileStage;
  constexpr int D = 128, PB = kTileWaves / HS, kStage = Stage::kBytes, kV = Stage::kV, kK = Stage::kK;
  const lds_addr lds0 = lds_address_of(smem_raw);
  const RowFragOffsets<D / 8> ro(lds0);
  const TrFragOffsets<D / 8, KSlots::kAccum> to(lds0);
  const int nrb = p.S / 32, slices = (p.Hq / p.Hkv) / HS, groups = slices * p.Hkv;
  const int group = blockIdx.x % groups, pull = blockIdx.x / groups;
  const int kvh = group % p.Hkv, slice = group / p.Hkv;
  // The group is the fast index, then (in launches of up to six rounds) the batch row, then the rank in the row's work-sorted
  // schedule. In larger ones sixteen tiles of a row go out together: an XCD then has a quarter of the rows' keys in use at a
  // time, which its L2 holds, and the tiles that come late are short either way. (8, 2048, 32/16), images, 268 / 243 us; (2, 13824,
  // 16/16), documents of 131 to 5665, 304 / 285; below, 0.91 to 1.1 times as fast by row: (6, 2304, 16/4) of 321 to 609, 53 / 54.
  int rank = pull / p.B, b = batch_row_of(pull, rank, p.B, groups);
  if (gridDim.x >= kRowsInTurnFrom) {
    const int tiles = nrb / PB, run = max(1, min(16, tiles / 4));
    const int turn = pull / (run * p.B), length = min(run, tiles - turn * run), at = pull - turn * run * p.B;
    b = at / length;
    rank = turn * run + at % length;
  }
  const int qt = uniform(meta_const(p.sched + query_schedule_offset(nrb, PB))[(size_t)b * schedule_ints(nrb) + rank]);
  const int w = uniform(threadIdx.x >> 6);
  const QueryWork<HS, kTileWaves> work(p, b, kvh, slice, qt);
  const size_t q_row_stride = (size_t)p.Hq * D, kv_row_stride = (size_t)p.Hkv * D;
  const size_t first_row = (size_t)b * p.S + work.rb * 32;
  const bf16* q_block = p.q + (first_row * p.Hq + work.h) * D;
  bf16* out_block = p.out + (first_row * p.Hq + work.h) * D;
  RowBlockLoader<D> q_rows;
  q_rows.request(q_block, q_row_stride);
  const QueryTileContext<D, HS, kTileWaves> ctx(p, b, kvh, slice, qt);  // (S is a multiple of 128: every tile is whole)
  const int last = ctx.last;
  if (ctx.first > last) {  // padding
    const int l = lane_id_here();
#pragma unroll
    for (int i = 0; i < 8; ++i)
      store_global16(out_block + (size_t)(4 * i + l / 16) * q_row_stride + l % 16 * 8, u32x4{0, 0, 0, 0});
    if (l < 32) p.lse[(first_row + l) * p.Hq + work.h] = 0.f;
    return;
  }

  const TileDma<kKeyTile, D / 8, kTileWaves * 64> dma(kv_row_stride * 2);
  const char* kbase = reinterpret_cast<const char*>(ctx.kbase);
  const char* vbase = reinterpret_cast<const char*>(ctx.vbase);
  const size_t tile_bytes = (size_t)kKeyTile * kv_row_stride * 2;
  auto issue_ids = [&](int tile) {
    if (threadIdx.x < 16) dma16_s(ctx.segb + tile * kKeyTile, threadIdx.x * 16, lds0 + Stage::seg_slot(tile));
  };
  auto issue_v = [&](int tile, lds_addr stage) { dma.issue(vbase + (size_t)tile * tile_bytes, stage + kV); };
  auto issue_k = [&](int tile, lds_addr stage) {
    dma.issue(kbase + (size_t)tile * tile_bytes, stage + kK);
    issue_ids(tile);
  };
  if (threadIdx.x == 0) lds_store<int>(lds0 + Stage::kLost, 0);

  for (bool careful = false;; careful = true) {  // (a second time where a row's sum was lost)
    int t = ctx.first;
    issue_k(t, lds0);
    issue_v(t, lds0);
    KeyTileBounds kb = key_tile_bounds(ctx.meta_b, t), nb = {0, 0, 0};  // bounds of tiles t and t + 1
    if (t + 1 <= last) nb = key_tile_bounds(ctx.meta_b, t + 1);
    bool visit = ctx.wave_visits(kb, t);  // does this wavefront see tile t (its scores are in the buffer of t)
    bool visit_prev = false;              // ... tile t - 1 (P^T in the other buffer, PV product still to do)

    // Which of the 64 tiles from `chart_base` on this wavefront sees, and sees in full (lane j: tile chart_base + j).
    int chart_base = 0;
    unsigned long long seen = 0, plain = 0;
    auto chart = [&](int base) {
      chart_base = base;
      const int tj = base + lane_id_here();
      bool sees = false, full = false;
      if (tj >= ctx.first && tj <= last) {
        const int* a = ctx.meta_b + (size_t)(2 * tj) * kMetaW;
        const int* c = a + kMetaW;
        const int a_min = a[kMinNz], c_min = c[kMinNz];
        const int k_min = a_min == 0 ? c_min : (c_min == 0 ? a_min : min(a_min, c_min));
        const int k_max = max(a[kMaxId], c[kMaxId]);
        const int k_uniform = (a[kUniform] == c[kUniform]) ? a[kUniform] : 0;
        sees = blocks_interact(ctx.mine.min_nz, ctx.mine.max_id, ctx.mine.end_max, k_min, k_max, tj * kKeyTile);
        full = sees && tile_is_interior(ctx.mine.uniform, ctx.mine.end_min, k_uniform, tj * kKeyTile + kKeyTile - 1);
      }
      seen = __ballot(sees);
      plain = __ballot(full);
    };
    chart(t - 1);
    bf16x8 qf[D / 16];
    q_rows.to_fragments(lds0 + (kStage + w * Stage::kPatchBytes), qf);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) qf[ks] = scale_bf16x8(qf[ks], p.scale);
    dma_wait_all();
    __syncthreads();
    if (t + 1 <= last) issue_k(t + 1, lds0 + kStage);  // (the Q rows are out of its place)
    float m_run = kNegInf;  // softmax reference (a recent running max), log2 domain
    float l_run = 0.f;      // this lane's share of the running sum
    bool lost = false;      // a sum of this wavefront is
    // (statement "b" writes buffer a: the first tile counts even)
    if (visit) fwd_qk_zero_b<kK>(ro, qf);
    else fwd_acc_zero();
    dma_wait_all();
    __builtin_amdgcn_s_barrier();

    auto must_rescale = [&](float mx) { return __any(mx > m_run + kRescaleSlack) != 0; };
    auto rescale = [&](float mx) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = exp2_fast(m_run - (m_new == kNegInf ? 0.f : m_new));
      l_run *= alpha;
      if (__any(m_run != kNegInf)) fwd_acc_scale(alpha);
      m_run = m_new;
    };
    // Sources of the copies that the statements of tile t's step issue (V of tile t, K two tiles on, or of tile `last` to where
    // nothing reads it), and this wavefront's place in a stage.
    unsigned long long v_source = 0, k_source = 0;
    const unsigned own = uniform((int)(unsigned)(uintptr_t)(lds0 + w * 1024));
    const auto scalar64 = [](const char* ptr) {
      const unsigned long long a = (unsigned long long)(uintptr_t)ptr;
      const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a);
      const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(a >> 32));
      return ((unsigned long long)hi << 32) | (unsigned long long)lo;
    };
    auto set_sources = [&] {
      v_source = scalar64(vbase + (size_t)t * tile_bytes);
      k_source = scalar64(kbase + (size_t)min(t + 2, last) * tile_bytes);
    };
    auto next_sources = [&] {
      v_source += tile_bytes;
      if (t + 3 <= last) k_source += tile_bytes;
    };
    auto end_of_step = [&] {
      dma_wait_all();  // stage t
      __builtin_amdgcn_s_barrier();
      ++t;
    };

    // PARITY = (t - first) & 1: the scores of tile t are in buffer a (0) or b (1), stage t - 1 (V(t - 1), K(t + 1)) is in LDS
    // buffer 1 - PARITY, stage t goes to PARITY. The statements of a step between two tiles that are seen, with the maximum:
    auto following_statements = [&](auto parity_tag) {
      constexpr int PARITY = decltype(parity_tag)::value;
      constexpr int V_OFF = (1 - PARITY) * kStage + kV, K_OFF = (1 - PARITY) * kStage + kK;
      if (t + 2 <= last) issue_ids(t + 2);
      float mx;
      if constexpr (PARITY == 0) mx = fwd_max_4_a<V_OFF>(to, v_source, k_source, dma.lane_off, own + kV, own + kK);
      else mx = fwd_max_4_b<V_OFF>(to, v_source, k_source, dma.lane_off, own + kStage + kV, own + kStage + kK);
      float psum = 0.f;
      if (must_rescale(mx)) {
        if constexpr (PARITY == 0) fwd_pv_late_a<V_OFF>(to);
        else fwd_pv_late_b<V_OFF>(to);
        rescale(mx);
        const float m_use = (m_run == kNegInf) ? 0.f : m_run;
        if constexpr (PARITY == 0) {
          fwd_exp_only_a(m_use, psum);
          fwd_qk_a<K_OFF>(ro, qf);
        } else {
          fwd_exp_only_b(m_use, psum);
          fwd_qk_b<K_OFF>(ro, qf);
        }
      } else {
        const float m_use = (m_run == kNegInf) ? 0.f : m_run;
        if constexpr (PARITY == 0) {
          fwd_exp_a_a<V_OFF>(to, m_use, psum);
          fwd_exp_b_a<K_OFF>(ro, qf, m_use, psum);
        } else {
          fwd_exp_a_b<V_OFF>(to, m_use, psum);
          fwd_exp_b_b<K_OFF>(ro, qf, m_use, psum);
        }
      }
      l_run += psum;
    };
    // The step of a tile seen in full between two that are seen, with the maximum, and without (every row has a reference):
    auto plain_step = [&](auto parity_tag) {
      following_statements(parity_tag);
      next_sources();
      end_of_step();
    };
    auto free_step = [&](auto parity_tag) {
      constexpr int PARITY = decltype(parity_tag)::value;
      constexpr int V_OFF = (1 - PARITY) * kStage + kV, K_OFF = (1 - PARITY) * kStage + kK;
      if (t + 2 <= last) issue_ids(t + 2);
      if constexpr (PARITY == 0) {
        fwd_free_pv_a<V_OFF>(to, v_source, k_source, dma.lane_off, own + kV, own + kK, m_run, l_run);
        fwd_free_qk_a<K_OFF>(ro, qf, m_run, l_run);
      } else {
        fwd_free_pv_b<V_OFF>(to, v_source, k_source, dma.lane_off, own + kStage + kV, own + kStage + kK, m_run, l_run);
        fwd_free_qk_b<K_OFF>(ro, qf, m_run, l_run);
      }
      next_sources();
      end_of_step();
    };
    // The step of any tile.
    auto step = [&](auto parity_tag) {
      constexpr int PARITY = decltype(parity_tag)::value;
      constexpr int V_OFF = (1 - PARITY) * kStage + kV, K_OFF = (1 - PARITY) * kStage + kK;
      const bool visit_next = t < last && ctx.wave_visits(nb, t + 1);
      const bool interleaved = visit_prev && visit && visit_next;
      if (!interleaved) {
        if (t != ctx.first) issue_v(t, lds0 + PARITY * kStage);  // (V(first) went with the first copies)
        if (t + 2 <= last) issue_k(t + 2, lds0 + PARITY * kStage);
      }
      if (visit) {
        // (a key tile with one shared id turns the id test into a per-query predicate)
        const int k_uniform = uniform(kb.uniform);
        const bool need_seg = ctx.mine.uniform == 0 || ctx.mine.uniform != k_uniform;
        const bool need_causal = t * kKeyTile + kKeyTile - 1 > ctx.mine.end_min;
        if (need_seg || need_causal) {
          const int seg_cmp = ctx.row_valid() ? ctx.seg_q : -1;
          const int half = lane_id_here() >> 5;
          const int rel = ctx.end_q - t * kKeyTile - 4 * half;
          if (k_uniform == 0) {
            const lds_addr ids = lds0 + (Stage::seg_slot(t) + 16 * half);
            if constexpr (PARITY == 0) fwd_mask_ids_a(ids, seg_cmp);
            else fwd_mask_ids_b(ids, seg_cmp);
            if (need_causal) {
              if constexpr (PARITY == 0) fwd_mask_causal_a(rel);
              else fwd_mask_causal_b(rel);
            }
          } else {
            const int rel_or_none = seg_cmp != k_uniform ? -1 : rel;
            if constexpr (PARITY == 0) fwd_mask_causal_a(rel_or_none);
            else fwd_mask_causal_b(rel_or_none);
          }
        }
      }
      if (interleaved) {
        set_sources();
        following_statements(parity_tag);
      } else {
        if (visit_prev) {
          if constexpr (PARITY == 0) fwd_pv_a<V_OFF>(to);
          else fwd_pv_b<V_OFF>(to);
        }
        if (visit) {
          float mx;
          if constexpr (PARITY == 0) mx = fwd_max_only_a();
          else mx = fwd_max_only_b();
          if (must_rescale(mx)) rescale(mx);
          const float m_use = (m_run == kNegInf) ? 0.f : m_run;
          float psum = 0.f;
          if constexpr (PARITY == 0) fwd_exp_only_a(m_use, psum);
          else fwd_exp_only_b(m_use, psum);
          l_run += psum;
        }
        if (visit_next) {
          if constexpr (PARITY == 0) fwd_qk_a<K_OFF>(ro, qf);
          else fwd_qk_b<K_OFF>(ro, qf);
        }
      }
      KeyTileWords ahead_words = key_tile_words_request(ctx.meta_b, min(t + 2, last));  // (they land under the wait below)
      end_of_step();
      key_tile_words_wait(ahead_words);
      visit_prev = visit;
      visit = visit_next;
      kb = nb;
      nb = key_tile_bounds(ahead_words);
    };

    constexpr std::integral_constant<int, 0> kEven{};
    constexpr std::integral_constant<int, 1> kOdd{};
    bool free_steps = !careful;
    while (t <= last) {
      // a stretch of plain steps from tile t on: tiles u with u - 1 seen, u plain, u + 1 seen
      if (t - chart_base >= 63) chart(t - 1);
      const unsigned long long stretch = ((seen << 1) & plain & (seen >> 1)) >> (t - chart_base);
      int n = (int)__builtin_ctzll(~stretch);
      const bool odd = ((t - ctx.first) & 1) != 0;
      if (n == 0) {
        if (odd) step(kOdd);
        else step(kEven);
        continue;
      }
      set_sources();
      if (!free_steps || __any(m_run == kNegInf)) {
        if (odd) plain_step(kOdd);
        else plain_step(kEven);
      } else {
        if (odd) {
          free_step(kOdd);
          --n;
        }
        for (; n >= 2; n -= 2) {
          free_step(kEven);
          free_step(kOdd);
          if (__any(!(l_run <= kFollowFromSum))) break;
        }
        if (n == 1) free_step(kEven);
        free_steps = !__any(!(l_run <= kFollowFromSum));
        if (!free_steps) lost = lost || __any(!(l_run <= kLostFromSum));
      }
      // back to the general step: tiles t - 1 and t are seen, and their bounds are read again
      visit_prev = true;
      visit = true;
      kb = key_tile_bounds(ctx.meta_b, t);
      nb = key_tile_bounds(ctx.meta_b, min(t + 1, last));
    }
    if (visit_prev) {  // (stage `last` is in LDS buffer (last - first) & 1, P^T(last) in the score buffer of that parity)
      if (((last - ctx.first) & 1) == 0) fwd_pv_b<kV>(to);
      else fwd_pv_a<kStage + kV>(to);
    }
    if (lost) lds_store<int>(lds0 + Stage::kLost, 1);
    __syncthreads();  // the stages become store patches
    const int again = lds_load<int>(lds0 + Stage::kLost);
    const float l_tot = pair_sum(l_run);
    const bool has = l_tot > 0.f;
    const float inv = has ? 1.f / l_tot : 0.f;
    const int le = lane_id_here();
    if (le < 32) p.lse[(first_row + le) * p.Hq + work.h] = has ? (__logf(l_tot) + m_run * kLn2) : 0.f;
    fwd_store_rows(inv, lds0 + w * Stage::kPatchBytes, out_block, q_row_stride);
    if (__builtin_expect(careful || uniform(again) == 0, 1)) return;
    __syncthreads();
    q_rows.request(q_block, q_row_stride);
  }
}

}  // namespace ct
