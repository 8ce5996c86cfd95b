// C ABI of the attention hot path: argument validation and launches.
#include <atomic>
#include <algorithm>
#include <type_traits>
#include <utility>

#include "ct_attn_bwd_kernels.hip.h"
#include "ct_attn_dkv_wide.hip.h"
#include "ct_attn_fwd_shares.hip.h"
#include "ct_attn_fwd_split.hip.h"
#include "ct_attn_fwd_tile.hip.h"
#include "ct_attn_kernels.hip.h"
#include "ct_error.h"
#include "ct_lanes.hip.h"

#include <string.h>

#include <initializer_list>

namespace ct {

// ---------------------------------------------------------------------------
// Tile bounds, in three launches, two for short rows, one for few positions: the summary of every 32-position block; from a
// row's summaries, what each block has to visit; from those ranges, the work-sorted schedules, the dS offsets and the bins.
//
// All of it is latency: the searches and the ranking are quadratic in a row's blocks, and one
// workgroup per row for everything took 43 us at S = 4096 and 0.6 ms at S = 32768 (its LDS pipe). Now
// 32 lanes read a block's ids, 16 lanes share the search of a block in a workgroup per 64 blocks, and
// every schedule has a workgroup of its own, with as many lanes per tile as there are threads for.
// ---------------------------------------------------------------------------

// Lanes that share one of n work items of a workgroup of `threads` (a power of two, at most 64).
CT_DEVICE int lanes_per_item(int n, int threads) {
  int lanes = 1;
  while (lanes < 64 && lanes * 2 * n <= threads) lanes *= 2;
  return lanes;
}
// What a block's record says of its ids and visible ends; 32 consecutive lanes per block, all of them get it.
struct BlockIds {
  int min_nz, max_id, uniform, end_min, end_max;
  CT_DEVICE BlockIds(const int* seg, const int* end, size_t row, int pos) {
    const int id = seg[row + pos], e = end ? end[row + pos] : pos;
    const bool counts = id != 0;
    const int low = min_over(counts ? id : INT_MAX, 32), high = max_over(counts ? id : INT_MIN, 32);
    end_min = min_over(counts ? e : INT_MAX, 32);
    end_max = max_over(counts ? e : -1, 32);
    const int zeros = 32 - __popcll(__ballot(counts) >> (threadIdx.x & 32) & 0xffffffffull);
    max_id = max(high, 0);
    min_nz = max_id == 0 ? 0 : low;  // reference: all-padding block -> (0, 0)
    uniform = zeros == 0 && low == high ? low : 0;
  }
  CT_DEVICE void store(int* m) const {
    m[kMinNz] = min_nz;
    m[kMaxId] = max_id;
    m[kUniform] = uniform;
    m[kEndMin] = end_min;
    m[kEndMax] = end_max;
    m[10] = 0;
    m[11] = 0;
  }
};

// What the searches read of the records of n blocks from position `first` on (of one row or of several, one behind the other):
// four lanes per block, eight positions each.
CT_DEVICE void search_records(const int* seg, const int* end, size_t first, int S, int n, int* min_nz, int* max_id, int* end_max) {
  const int nrb = S / 32, quarter = threadIdx.x % 4;
  for (int i0 = threadIdx.x / 4; i0 < n; i0 += 512) {  // (n is a multiple of 4: whole rows of 16 lanes)
    int id[2][8], e[2][8];  // two blocks in flight
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const size_t at = first + (size_t)(i0 + 256 * j < n ? i0 + 256 * j : i0) * 32 + quarter * 8;
      __builtin_memcpy(id[j], seg + at, sizeof id[j]);
      if (end) __builtin_memcpy(e[j], end + at, sizeof e[j]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = i0 + 256 * j;
      if (i >= n) break;
      const int pos = i % nrb * 32 + quarter * 8;
      int low = INT_MAX, high = 0, last = -1;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const bool counts = id[j][k] != 0;
        low = min(low, counts ? id[j][k] : INT_MAX);
        high = max(high, id[j][k]);
        last = max(last, counts ? (end ? e[j][k] : pos + k) : -1);
      }
      low = min_over(low, 4);
      high = max_over(high, 4);
      last = max_over(last, 4);
      if (quarter == 0) {
        min_nz[i] = high == 0 ? 0 : low;
        max_id[i] = high;
        end_max[i] = last;
      }
    }
  }
}

// grid (ceil(S / 1024), B)
__global__ __launch_bounds__(1024) void attn_blocks_kernel(const int* seg, const int* end, int S, int* meta) {
  const int b = blockIdx.y, pos = blockIdx.x * 1024 + threadIdx.x;
  if (pos >= S) return;  // (S % 128 == 0: whole wavefronts)
  const BlockIds block(seg, end, (size_t)b * S, pos);
  if (pos % 32 == 0) block.store(meta + ((size_t)b * (S / 32) + pos / 32) * kMetaW);
}

// Block summaries in the reference's format (ct_attn_block_summary); `block` = 0: none.
struct SummaryOut {
  int* out;
  int block, width;  // width 3: with the largest visible end
};

// 16 lanes share the search of a block: the first and last 64-key tile that row block rb has to visit as queries, and the first
// and last 32-row query block that it is visited by as keys; all of the lanes get them.
constexpr int kSearchLanes = 16;
struct VisitRange {
  int first = INT_MAX, last = -1;
  CT_DEVICE void add(int i) {
    first = min(first, i);
    last = i;
  }
  CT_DEVICE void over_lanes() {
    first = min_over(first, kSearchLanes);
    last = max_over(last, kSearchLanes);
  }
};
template <class MinNz, class MaxId, class EndMax>
CT_DEVICE VisitRange visited_tiles(MinNz min_nz, MaxId max_id, EndMax end_max, int S, int rb, int lane) {
  VisitRange range;
  const int my_min = min_nz(rb), my_max = max_id(rb), my_end = end_max(rb);
  if (my_min != 0) {
    const int t_hi = min(my_end / kKeyTile, S / kKeyTile - 1);
    for (int t = lane; t <= t_hi; t += kSearchLanes) {
      const int a_min = min_nz(2 * t), c_min = min_nz(2 * t + 1);
      const int k_min = a_min == 0 ? c_min : (c_min == 0 ? a_min : min(a_min, c_min));
      const int k_max = max(max_id(2 * t), max_id(2 * t + 1));
      if (blocks_interact(my_min, my_max, my_end, k_min, k_max, t * kKeyTile)) range.add(t);
    }
  }
  range.over_lanes();
  return range;
}
template <class MinNz, class MaxId, class EndMax>
CT_DEVICE VisitRange visiting_blocks(MinNz min_nz, MaxId max_id, EndMax end_max, int S, int rb, int lane) {
  VisitRange range;
  const int my_min = min_nz(rb), my_max = max_id(rb);
  if (my_min != 0)
    for (int qb = lane; qb < S / 32; qb += kSearchLanes)
      if (blocks_interact(min_nz(qb), max_id(qb), end_max(qb), my_min, my_max, rb * 32)) range.add(qb);
  range.over_lanes();
  return range;
}

// grid (ceil(nrb / 64), B): 16 lanes per block search what it has to visit; the workgroups of a row also
// write its block summaries. With `seg` every workgroup forms the records of its whole row by itself and stores its
// own: a launch and its latency less than with attn_blocks_kernel in front, for rows of up to kFusedRows positions
// (8 loads per thread). Both sides, us: [4, 4096] 4.1 + 4.2 / 5.5, [8, 8192] 4.3 + 5.1 / 8.5, [4, 16384] 4.3 + 8.2 / 14.6,
// [1, 32768] 4.1 + 14.0 / 25.1.
constexpr int kFusedRows = 8192;
// LDS is compiled apart: one pointer to either kind of memory makes every access a flat one ([4, 16384] 13.8 -> 8.2 us,
// [1, 32768] 25.1 -> 14.0).
template <bool LDS>
CT_DEVICE void build_ranges(int* meta, int S, const SummaryOut& queries, const SummaryOut& keys, const int* seg, const int* end,
                            int part, int parts, int b, int* lds_rows) {  // lds_rows [3][nrb]: min_nz, max_id, end_max
  const int nrb = S / 32;
  int* mb = meta + (size_t)b * nrb * kMetaW;
  if (LDS && seg) {
    search_records(seg, end, (size_t)b * S, S, nrb, lds_rows, lds_rows + nrb, lds_rows + 2 * nrb);
    for (int pos = part * 2048 + threadIdx.x; pos < min(S, (part + 1) * 2048); pos += 1024) {  // (S % 128 == 0: whole wavefronts)
      const BlockIds block(seg, end, (size_t)b * S, pos);
      if (pos % 32 == 0) block.store(mb + pos / 32 * kMetaW);
    }
    __syncthreads();
  } else if (LDS) {
    for (int i = threadIdx.x; i < nrb; i += 1024) {
      lds_rows[i] = mb[i * kMetaW + kMinNz];
      lds_rows[nrb + i] = mb[i * kMetaW + kMaxId];
      lds_rows[2 * nrb + i] = mb[i * kMetaW + kEndMax];
    }
    __syncthreads();
  }
  auto min_nz = [&](int i) { return LDS ? lds_rows[i] : mb[i * kMetaW + kMinNz]; };
  auto max_id = [&](int i) { return LDS ? lds_rows[nrb + i] : mb[i * kMetaW + kMaxId]; };
  auto end_max = [&](int i) { return LDS ? lds_rows[2 * nrb + i] : mb[i * kMetaW + kEndMax]; };

  constexpr int kLanes = kSearchLanes;
  const int lane = threadIdx.x % kLanes, rb = part * (1024 / kLanes) + threadIdx.x / kLanes;
  if (rb < nrb) {
    const VisitRange tiles = visited_tiles(min_nz, max_id, end_max, S, rb, lane);
    const VisitRange blocks = visiting_blocks(min_nz, max_id, end_max, S, rb, lane);
    if (lane == 0) {
      int* m = mb + rb * kMetaW;
      m[kKvFirst] = tiles.first;
      m[kKvLast] = tiles.last;
      m[kQFirst] = blocks.first;
      m[kQLast] = blocks.last;
    }
  }

  for (int side = 0; side < 2; ++side) {
    const SummaryOut& summary = side ? keys : queries;
    if (!summary.block) continue;
    const int per = summary.block / 32, count = S / summary.block, groups = 1024 / kLanes;
    for (int i = part * groups + threadIdx.x / kLanes; i < count; i += parts * groups) {
      int low = INT_MAX, high = 0, last = 0;
      for (int k = i * per + lane; k < (i + 1) * per; k += kLanes) {
        if (min_nz(k) != 0) low = min(low, min_nz(k));
        high = max(high, max_id(k));
        last = max(last, end_max(k));
      }
      low = min_over(low, kLanes);
      high = max_over(high, kLanes);
      last = max_over(last, kLanes);
      if (lane == 0) {
        int* out = summary.out + ((size_t)b * count + i) * summary.width;
        out[0] = high == 0 ? 0 : low;
        out[1] = high;
        if (summary.width == 3) out[2] = last;
      }
    }
  }
}
template <bool LDS>
__global__ __launch_bounds__(1024) void attn_ranges_kernel(int* meta, int S, SummaryOut queries, SummaryOut keys,
                                                           const int* seg, const int* end) {
  extern __shared__ __align__(16) int lds_rows[];
  build_ranges<LDS>(meta, S, queries, keys, seg, end, blockIdx.x, gridDim.x, blockIdx.y, lds_rows);
}

// The working arrays are in LDS or, for rows beyond 262144 positions and for many tiles, in the metadata buffer's
// scratch region. In LDS a tile's work and its index are one key, larger for more work and, at the same work, for the lower
// index (work is below 2^17 there), and a comparison is two instructions. The LDS form
// is compiled apart: through pointers that may be either, every access waits for the vector memory's counter too.
template <bool LDS>
struct TileWork {
  static constexpr int kIndexBits = 14;
  static_assert(kPrepareLdsRowBlocks <= 1 << kIndexBits && kBinsLdsInts / 3 <= 1 << kIndexBits, "tiles that the keys tell apart");
  CT_DEVICE static int pack(int work, int i) { return LDS ? (work << kIndexBits) + (1 << kIndexBits) - 1 - i : work; }
  CT_DEVICE static int work(int key) { return LDS ? key >> kIndexBits : key; }
};
// Number of the tiles in front of tile i when they are ordered by decreasing work, ties by index;
// shared by `lanes` lanes. Read in 16-byte quads from the first multiple of 16 bytes on: the arrays in LDS start
// at one, those in the scratch region anywhere.
template <bool LDS>
CT_DEVICE int rank_of(const int* w, int n, int i, int lanes) {
  const int wi = w[i], lane = threadIdx.x % lanes;
  const int head = LDS ? 0 : min(n, (int)(-(uintptr_t)w / sizeof(int) % 4)), quads = (n - head) / 4;
  int rank = 0;
  auto count = [&](int wv, int k) { rank += LDS ? wv > wi : (wv > wi) || (wv == wi && k < i); };
  for (int k = lane; k < head; k += lanes) count(w[k], k);
  for (int q = lane; q < quads; q += lanes) {
    const int4 v = reinterpret_cast<const int4*>(w + head)[q];
    const int k = head + 4 * q;
    count(v.x, k);
    count(v.y, k + 1);
    count(v.z, k + 2);
    count(v.w, k + 3);
  }
  for (int k = head + 4 * quads + lane; k < n; k += lanes) count(w[k], k);
  return sum_over(rank, lanes);
}
// What the row blocks of a row have to visit, as queries (64-key tiles) or as keys (32-row query blocks): from the table ...
struct TableRanges {
  const int* row;
  int from;  // kKvFirst or kQFirst, followed by the last
  CT_DEVICE int first(int rb) const { return row[rb * kMetaW + from]; }
  CT_DEVICE int last(int rb) const { return row[rb * kMetaW + from + 1]; }
};
// ... or from LDS, where a workgroup has searched them by itself.
struct LocalRanges {
  const int *firsts, *lasts;
  CT_DEVICE int first(int rb) const { return firsts[rb]; }
  CT_DEVICE int last(int rb) const { return lasts[rb]; }
};
// Tiles between the first and the last that row blocks first .. end - 1 have to visit.
template <class Ranges>
CT_DEVICE int visit_span(const Ranges& ranges, int first_block, int end_block) {
  int first = INT_MAX, last = -1;
  for (int k = first_block; k < end_block; ++k) {
    first = min(first, ranges.first(k));
    last = max(last, ranges.last(k));
  }
  return last >= first ? last - first + 1 : 0;
}

// One of the five schedules of a batch row: query tiles of 1, 2, 4 row blocks, 128-key tiles, query
// tiles of 8.
// (`ranges`: the row's, as keys for job 3, else as queries)
template <bool LDS, class Ranges>
CT_DEVICE void build_schedule(int job, const Ranges& ranges, int nrb, int* sched, int* work) {
  const int pb = job == 3 ? 4 : job == 4 ? 8 : 1 << job, n = job == 4 ? (nrb + 7) / 8 : nrb / pb;
  for (int i = threadIdx.x; i < n; i += 1024)
    work[i] = TileWork<LDS>::pack(visit_span(ranges, i * pb, min(nrb, (i + 1) * pb)), i);
  __syncthreads();
  const int lanes = lanes_per_item(n, 1024);
  int* out = sched + (job == 3 ? key_schedule_offset(nrb) : query_schedule_offset(nrb, pb));
  for (int i = threadIdx.x / lanes; i < n; i += 1024 / lanes) {
    const int rank = rank_of<LDS>(work, n, i, lanes);
    if (threadIdx.x % lanes == 0) out[rank] = i;
  }
}

// Where the dS blocks of each key block of a row start (kDsOff): exclusive prefix sum of the lengths of
// the query-block ranges. Every thread sums a contiguous run of row blocks, the runs are
// scanned across the workgroup, and each thread then walks its run again.
template <class Ranges>
CT_DEVICE void build_ds_offsets(const Ranges& ranges, int* mb, int nrb) {
  __shared__ long long wave_sum[16];
  const int per = (nrb + 1023) / 1024, lane = threadIdx.x & 63;
  const int lo = min(nrb, (int)threadIdx.x * per), hi = min(nrb, lo + per);
  long long local = 0;
  for (int rb = lo; rb < hi; ++rb) local += visit_span(ranges, rb, rb + 1);
  long long incl = local;
  for (int off = 1; off < 64; off <<= 1) {
    const long long below = __shfl_up(incl, off, 64);
    if (lane >= off) incl += below;
  }
  if (lane == 63) wave_sum[threadIdx.x >> 6] = incl;
  __syncthreads();
  long long run = incl - local;
  for (int k = 0; k < (int)threadIdx.x >> 6; ++k) run += wave_sum[k];
  for (int rb = lo; rb < hi; ++rb) {
    mb[rb * kMetaW + kDsOff] = (int)min(run, (long long)INT_MAX);
    run += visit_span(ranges, rb, rb + 1);
  }
}

// Lane moves of 32 or 64 bits: the value of the lane that DPP control `CONTROL` names, all ones where it names none or the
// row of 16 lanes is not in ROWS; lane k's value, as a scalar; the value sent to lane `to`.
template <int CONTROL, int ROWS>
CT_DEVICE unsigned moved_lanes(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, CONTROL, ROWS, 0xf, false);
}
template <int CONTROL, int ROWS>
CT_DEVICE unsigned long long moved_lanes(unsigned long long v) {
  return (unsigned long long)moved_lanes<CONTROL, ROWS>((unsigned)(v >> 32)) << 32 | moved_lanes<CONTROL, ROWS>((unsigned)v);
}
// How many of the first 32 lanes hold less. Keys below 2^31: the sign of a difference, of which no scalar register is
// part (a comparison's mask costs wait states on its way to the sum); lane moves reach the 15 others of a row of 16,
// and those of the other row once it has changed places.
template <int ROTATE>
CT_DEVICE unsigned rotated_below(unsigned other, unsigned v) {
  return ((unsigned)__builtin_amdgcn_mov_dpp((int)other, 0x120 + ROTATE, 0xf, 0xf, true) - v) >> 31;
}
template <int... ROTATE>
CT_DEVICE int rank_among(unsigned v, std::integer_sequence<int, ROTATE...>) {
  const unsigned across = (unsigned)__shfl_xor((int)v, 16, 64);
  return (int)(((across - v) >> 31) + ... + (rotated_below<ROTATE + 1>(v, v) + rotated_below<ROTATE + 1>(across, v)));
}
CT_DEVICE int rank_among(unsigned v) { return rank_among(v, std::make_integer_sequence<int, 15>{}); }
CT_DEVICE int rank_among(unsigned long long v) {
  int rank = 0;
  for (int k = 0; k < 32; ++k) {
    const unsigned low = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, k);
    const unsigned high = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), k);
    rank += ((unsigned long long)high << 32 | low) < v;
  }
  return rank;
}
CT_DEVICE unsigned sent_to(unsigned v, int to) { return (unsigned)__builtin_amdgcn_ds_permute(to * 4, (int)v); }
CT_DEVICE unsigned long long sent_to(unsigned long long v, int to) {
  return (unsigned long long)sent_to((unsigned)(v >> 32), to) << 32 | sent_to((unsigned)v, to);
}

// Packs the query tiles of the whole batch into kBins bins of near equal work
// (longest processing time first: the heaviest tile left goes to the least loaded bin, ties to the
// lowest bin), by one workgroup per tile size pb (2, 4, 8 row blocks). lds_bins: 3 ints per tile.
//
// The greedy pass is serial, but up to kBins of its steps can be taken together: with the bins ranked
// by load, the next tiles go to the bins of rank 0, 1, 2, ... until one of those just filled would
// again be the least loaded. Lane k of one wavefront holds the bin of rank k (its load and number as one key); a round of up
// to 32 tiles is a chain of some 800 clocks: 32 comparisons for the ranks, one exchange through LDS, a running minimum by lane
// moves. Nine rounds at four rows of 4096 (256 tiles); with shuffles, unpacked loads and arrays behind generic pointers a
// round took 2500 and the kernel 15.2 us, now 8.0.
// `ranges_of(b)`: what the row blocks of batch row b have to visit as queries.
template <bool LDS, class RangesOf>
CT_DEVICE void build_bins(int* meta, int B, int S, int pb, int* lds_bins, RangesOf ranges_of) {
  typedef std::conditional_t<LDS, unsigned, unsigned long long> Key;
  __shared__ int start[kBins + 1];
  const int nrb = S / 32;
  const int tpr = bin_tiles_per_row(nrb, pb), n = B * tpr;
  int* work = lds_bins;
  int* order = lds_bins + n;
  int* place = lds_bins + 2 * n;  // first the work in rank order, then (position in its bin) * kBins + bin
  int* region = meta + bin_region_offset(B, nrb, pb);
  for (int i = threadIdx.x; i < n; i += 1024) {
    const int b = i / tpr, qt = i % tpr;
    // a tile without keys still costs a launch of the prologue; +3 ~ prologue and store
    work[i] = TileWork<LDS>::pack(visit_span(ranges_of(b), qt * pb, min(nrb, (qt + 1) * pb)) + 3, i);
  }
  __syncthreads();
  const int lanes = lanes_per_item(n, 1024);
  for (int i = threadIdx.x / lanes; i < n; i += 1024 / lanes) {
    const int rank = rank_of<LDS>(work, n, i, lanes);
    if (threadIdx.x % lanes == 0) {
      order[rank] = i;
      place[rank] = TileWork<LDS>::work(work[i]);
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    // of the bin of rank `lane`: load * kBins + bin, and its number of tiles (lanes from kBins on keep out)
    Key key = lane < kBins ? (Key)lane : ~(Key)0;
    int count = 0;
    for (int r = 0; r < n;) {
      const int weight = r + lane < n ? place[r + lane] : 0;
      const Key filled = key + (Key)weight * kBins;
      // the least filled bin among those of lower rank
      Key least = lane < kBins ? filled : ~(Key)0;
      const auto step = [&](auto control, auto rows) {
        const Key other = moved_lanes<control.value, rows.value>(least);
        least = other < least ? other : least;
      };
      step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});  // from 1, 2, 4, 8 lanes below
      step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
      step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
      step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
      step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // lane 15 to the next sixteen
      least = moved_lanes<0x138, 0xf>(least);                                          // one lane up
      const unsigned long long stop = __ballot(lane >= kBins || r + lane >= n || least < key);
      const int taken = __ffsll(stop) - 1;  // at least one: nothing is below rank 0
      if (lane < taken) {
        key = filled;
        place[r + lane] = count * kBins + (int)(key % kBins);
        ++count;
      }
      r += taken;
      const int rank = lane < kBins ? rank_among(key) : lane;
      key = sent_to(key, rank);
      count = __builtin_amdgcn_ds_permute(rank * 4, count);
    }
    // back to lane = bin
    count = __builtin_amdgcn_ds_permute(lane < kBins ? (int)(key % kBins) * 4 : lane * 4, count);
    const int incl = wave_scan(count);
    if (lane < kBins) {
      start[lane] = incl - count;
      if (lane == kBins - 1) start[kBins] = incl;
    }
  }
  __syncthreads();
  // in rank order inside a bin: heaviest first
  if (threadIdx.x <= kBins) region[threadIdx.x] = start[threadIdx.x];
  for (int r = threadIdx.x; r < n; r += 1024)
    region[kBins + 1 + start[place[r] % kBins] + place[r] / kBins] = order[r];
}

// grid: the bins' three workgroups (they take longest), then six per batch row: its schedules and dS
// offsets. Working arrays in LDS when they fit, else in the scratch region of the metadata buffer.
__global__ __launch_bounds__(1024) void attn_schedules_kernel(int* meta, int B, int S, int* sched_all, int* row_scratch,
                                                              int* bins_scratch) {
  extern __shared__ __align__(16) int lds_work[];
  const int nrb = S / 32;
  if (blockIdx.x < 3) {
    const int pb = 2 << blockIdx.x;
    const auto ranges_of = [&](int b) { return TableRanges{meta + (size_t)b * nrb * kMetaW, kKvFirst}; };
    if (bins_scratch) build_bins<false>(meta, B, S, pb, bins_scratch + (size_t)blockIdx.x * 3 * B * bin_tiles_per_row(nrb, 2), ranges_of);
    else build_bins<true>(meta, B, S, pb, lds_work, ranges_of);
    return;
  }
  const int b = (blockIdx.x - 3) / 6, job = (blockIdx.x - 3) % 6;
  int* mb = meta + (size_t)b * nrb * kMetaW;
  const TableRanges ranges = {mb, job == 3 || job == 5 ? kQFirst : kKvFirst};
  if (job == 5) {
    build_ds_offsets(ranges, mb, nrb);
  } else {
    const int offset = job == 3 ? key_schedule_offset(nrb) : query_schedule_offset(nrb, job == 4 ? 8 : 1 << job);
    int* sched = sched_all + (size_t)b * schedule_ints(nrb);
    if (row_scratch) build_schedule<false>(job, ranges, nrb, sched, row_scratch + (size_t)b * 3 * nrb + offset);
    else build_schedule<true>(job, ranges, nrb, sched, lds_work);
  }
}

// Ranges, schedules, offsets and bins in one launch: a workgroup that needs the ranges of a row (or, for the bins, of all
// rows) forms the records and searches them by itself, the one side that it needs. That repeats work on compute units that have
// none, and saves a launch and the wait between two. grid: the bins' three workgroups, six per batch row, then build_ranges' ones.
// LDS, ints: 3 + 2 per row block that a workgroup searches, then its working arrays. Us of GPU time, two launches / one, and 2.3
// of the host's: [1, 128] 6.6 / 3.9, [2, 1024] 7.7 / 4.5, [1, 8192] 13.0 / 11.5, [3, 2944] 10.4 / 9.1. The bins' workgroups search
// the whole batch: with four rows or more the GPU's times meet at 9216 positions (4 to 12 rows 9.6 / 9.6, 9.1 / 9.1) and from
// 10240 on one launch is the longer one by less than the host saves ([4, 2560] 9.8 / 10.2, [3, 4096] 11.7 / 12.2, [12, 1024] 9.8 /
// 10.8, [96, 128] 9.5 / 10.8). Past the lines it is that, or a long row's search, by as much or more: [4, 4096] 13.1 / 14.0 (a
// batch's preparation as a whole 28.2 / 30.0 where the host keeps ahead), [1, 12160] 17.4 / 20.3. (A wavefront per row block with
// a key tile per lane and a ballot: a chain of LDS reads per block, [4, 4096] 19.7.)
constexpr int kOneLaunchPositions = 12288;
__global__ __launch_bounds__(1024) void attn_prepare_kernel(int* meta, int B, int S, SummaryOut queries, SummaryOut keys,
                                                            const int* seg, const int* end, int* sched_all) {
  extern __shared__ __align__(16) int lds[];
  const int nrb = S / 32, parts = (nrb + 63) / 64;
  int index = blockIdx.x;
  if (index >= 3 + 6 * B) {
    index -= 3 + 6 * B;
    build_ranges<true>(meta, S, queries, keys, seg, end, index % parts, parts, index / parts, lds);
    return;
  }
  const bool bins = index < 3;
  const int job = bins ? 0 : (index - 3) % 6, row0 = bins ? 0 : (index - 3) / 6, rows = bins ? B : 1, n = rows * nrb;
  const bool as_keys = job == 3 || job == 5;
  int *mins = lds, *maxs = lds + n, *ends = lds + 2 * n, *firsts = lds + 3 * n, *lasts = lds + 4 * n, *work = lds + 5 * n;
  search_records(seg, end, (size_t)row0 * S, S, n, mins, maxs, ends);
  __syncthreads();
  const int lane = threadIdx.x % kSearchLanes;
  for (int i = threadIdx.x / kSearchLanes; i < n; i += 1024 / kSearchLanes) {
    const int first_of_row = i / nrb * nrb;
    const auto min_nz = [&](int k) { return mins[first_of_row + k]; };
    const auto max_id = [&](int k) { return maxs[first_of_row + k]; };
    const auto end_max = [&](int k) { return ends[first_of_row + k]; };
    const VisitRange range = as_keys ? visiting_blocks(min_nz, max_id, end_max, S, i - first_of_row, lane)
                                     : visited_tiles(min_nz, max_id, end_max, S, i - first_of_row, lane);
    if (lane == 0) {
      firsts[i] = range.first;
      lasts[i] = range.last;
    }
  }
  __syncthreads();
  const LocalRanges ranges = {firsts, lasts};
  if (bins) {
    build_bins<true>(meta, B, S, 2 << index, work, [&](int b) { return LocalRanges{firsts + b * nrb, lasts + b * nrb}; });
  } else if (job == 5) {
    build_ds_offsets(ranges, meta + (size_t)row0 * nrb * kMetaW, nrb);
  } else {
    build_schedule<true>(job, ranges, nrb, sched_all + (size_t)row0 * schedule_ints(nrb), work);
  }
}

// One wavefront per block.
__global__ __launch_bounds__(256) void attn_block_summary_kernel(const int* seg, const int* end, int block,
                                                                 int nblocks, int width, int* out) {
  const int gid = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (gid >= nblocks) return;
  const size_t first = (size_t)gid * block;
  int low = INT_MAX, high = 0, last = 0;
  for (int i = lane; i < block; i += 64) {
    const int id = seg[first + i];
    if (id != 0) {
      low = min(low, id);
      high = max(high, id);
      if (end) last = max(last, end[first + i]);
    }
  }
  low = min_over(low, 64);
  high = max_over(high, 64);
  last = max_over(last, 64);
  if (lane != 0) return;
  out[(size_t)gid * width + 0] = high == 0 ? 0 : low;
  out[(size_t)gid * width + 1] = high;
  if (end) out[(size_t)gid * width + 2] = last;
}

static float round_to_bf16(float x) {
  uint32_t u;
  ::memcpy(&u, &x, 4);
  const uint32_t lsb = (u >> 16) & 1u;
  u += 0x7fffu + lsb;
  u &= 0xffff0000u;
  float y;
  ::memcpy(&y, &u, 4);
  return y;
}

static int validate_shape(const char* fn, int B, int S, int Hq, int Hkv, int D) {
  CT_REQUIRE(B > 0 && S > 0 && Hq > 0 && Hkv > 0, "%s: dimensions must be positive", fn);
  CT_REQUIRE(S % 128 == 0, "%s: sequence length %d has no 128-aligned tiling", fn, S);
  CT_REQUIRE(Hq % Hkv == 0,
             "%s: query head count must be divisible by the KV head count, got Hq=%d, Hkv=%d", fn,
             Hq, Hkv);
  if (D != 64 && D != 128) return fail(CT_UNSUPPORTED, "%s: head_dim must be 64 or 128, got %d", fn, D);
  // (block tables and work lists index 32-position blocks of the whole batch with 32-bit ints)
  if ((long long)B * S > (1ll << 26))
    return fail(CT_UNSUPPORTED, "%s: batch %d x sequence %d exceeds 2^26 positions", fn, B, S);
  // (the tile ranking of ct_attn_prepare is quadratic in the row blocks of one batch row: rows up to
  // 2^20 positions are what it is built and tested for)
  if (S > (1 << 20))
    return fail(CT_UNSUPPORTED, "%s: sequence %d exceeds 2^20 positions per batch row", fn, S);
  return CT_OK;
}

// Tiles move by 16-byte asynchronous copies, so every tensor base must be 16-byte aligned.
static bool aligned16(std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
  return true;
}

// Query heads of one KV head handled by a single workgroup.
static int heads_per_group(int Hq, int Hkv) {
  const int g = Hq / Hkv;
  return g % 4 == 0 ? 4 : (g % 2 == 0 ? 2 : 1);
}

// Kernels that need more than the default 64 KB of dynamic LDS say so once per kernel and device
// (the attribute belongs to the loaded code object of that device), not on every launch.
static int ensure_lds(const char* fn, const void* kernel, size_t bytes, std::atomic<unsigned>& done) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 32) device = -1;
  if (device >= 0 && (done.load(std::memory_order_acquire) >> device & 1u)) return CT_OK;
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess) return fail(CT_LAUNCH_FAILED, "%s: %s", fn, hipGetErrorString(e));
  if (device >= 0) done.fetch_or(1u << device, std::memory_order_release);
  return CT_OK;
}
#define CT_ENSURE_LDS(fn, kernel, bytes)                                                  \
  do {                                                                                    \
    static std::atomic<unsigned> done_{0};                                                \
    int rc_ = ensure_lds(fn, reinterpret_cast<const void*>(kernel), (bytes), done_);      \
    if (rc_) return rc_;                                                                  \
  } while (0)

// Workgroups that share a work bin of a (head slice, KV head) group. A workgroup fills a compute
// unit, so groups x 32 bins fill the 256 units whole times exactly when the groups come in eights;
// the fewest members that make (groups x members) a multiple of 8 do the same for every other count.
static int fwd_members(int groups) { return groups % 8 == 0 ? 1 : groups % 4 == 0 ? 2 : groups % 2 == 0 ? 4 : 8; }

template <int D, int HS>
static int launch_fwd(hipStream_t stream, const AttnParams& p) {
  const size_t smem = VkStage<D>::kTotalBytes;
  CT_ENSURE_LDS("ct_attn_fwd", (&attn_fwd_kernel<D, HS>), smem);
  const int groups = p.Hq / HS;  // (head slice, KV head)
  const int grid = groups * kBins * fwd_members(groups);
  LaunchScope scope1("attn_fwd_kernel", stream);
  hipLaunchKernelGGL((attn_fwd_kernel<D, HS>), dim3(grid), dim3(kFwdWaves * 64), smem, stream, p);
  return scope1.done();
}

template <int HS>
static int launch_fwd_tile(hipStream_t stream, const AttnParams& p) {
  CT_ENSURE_LDS("ct_attn_fwd", (&attn_fwd_tile_kernel<HS>), FwdTileStage::kTotalBytes);
  const int grid = (p.Hq / HS) * p.B * (p.S / 32 / (kTileWaves / HS));
  LaunchScope scope("attn_fwd_tile_kernel", stream);
  hipLaunchKernelGGL(attn_fwd_tile_kernel<HS>, dim3(grid), dim3(kTileWaves * 64), FwdTileStage::kTotalBytes, stream, p);
  return scope.done();
}

template <int D, int NW>
static int launch_fwd_shares(hipStream_t stream, const AttnParams& p) {
  const size_t smem = NW * ShareRegion<D>::kBytes;
  CT_ENSURE_LDS("ct_attn_fwd", (&attn_fwd_shares_kernel<D, NW>), smem);
  LaunchScope scope("attn_fwd_shares_kernel", stream);
  hipLaunchKernelGGL((attn_fwd_shares_kernel<D, NW>), dim3(p.Hq * p.B * (p.S / 32)), dim3(NW * 64), smem, stream, p);
  return scope.done();
}

template <int D, int HS, int NW, int KS, int KB, int SUB>
static int launch_fwd_split(hipStream_t stream, const AttnParams& p) {
  const size_t smem = SplitStage<D, NW, KS, KB, SUB>::kTotalBytes;
  CT_ENSURE_LDS("ct_attn_fwd", (&attn_fwd_split_kernel<D, HS, NW, KS, KB, SUB>), smem);
  const int grid = (p.Hq / HS) * p.B * bin_tiles_per_row(p.S / 32, NW / KS / HS);
  LaunchScope scope("attn_fwd_split_kernel", stream);
  hipLaunchKernelGGL((attn_fwd_split_kernel<D, HS, NW, KS, KB, SUB>), dim3(grid), dim3(NW * 64), smem, stream, p);
  return scope.done();
}
template <int D, int NW, int KS, int KB, int SUB>
static int launch_fwd_split(hipStream_t stream, const AttnParams& p) {
  const int hs = heads_per_group(p.Hq, p.Hkv);
  if constexpr (NW / KS >= 4)
    if (hs == 4) return launch_fwd_split<D, 4, NW, KS, KB, SUB>(stream, p);
  if constexpr (NW / KS >= 2)
    if (hs >= 2) return launch_fwd_split<D, 2, NW, KS, KB, SUB>(stream, p);
  return launch_fwd_split<D, 1, NW, KS, KB, SUB>(stream, p);
}

// By the row blocks of the launch (32 query rows of one head: one wavefront's work; the device has
// 1024 SIMDs). Few of them leave SIMDs idle while the longest row's chain of steps runs: its keys
// are then shared by wavefronts. Where the lines lie was measured over row lengths 128 to 26496 and
// documents from 36 positions to the whole row:
//   few row blocks: attn_fwd_shares_kernel as long as all its workgroups are on the device at once, two on a compute unit with
//     four wavefronts at head dimension 128, four at 64. Past that short documents pay for a second round (128: [2, 4480, 2/2],
//     560 row blocks, images 66 / 40 but documents of 32 to 64 positions 9.5 / 11.4; 64: [1, 3456, 8/2], 864, 7.6 / 8.0), and in
//     rows below 512 positions there is little to share. Eight wavefronts, half as many on a compute unit, pay from 1024
//     positions on up to 256 and 512 row blocks (by four / eight: [1, 8192, 1/1, 128] 65 / 44, [1, 4096, 4/4, 64] 27 / 22,
//     documents of 100 to 200 there 7.6 / 8.0; [1, 4096, 4/4, 128], 512 row blocks, such documents 8.7 / 12.6).
//     Head dimension 64 from 513 row blocks on, 57 shapes, time here over that by two wavefronts with shared stages: documents
//     of 256 to 900 0.70 to 0.91, whole rows 0.56 to 0.95, 100 to 200 0.86 to 1.02. Documents of 16 to 64 take 0.94 to 1.01
//     where each head has stages of its own either way (up to 544 row blocks 0.98 to 1.11), and 1.06 to 1.13, half a
//     microsecond, where two or four heads could share them ([1, 2176, 8/4] 6.1 -> 6.8, but whole rows 23.8 -> 16.6).
//     Three wavefronts at head dimension 128 (three workgroups on a compute unit, 768 at once) where every head has its own
//     keys, in rows of 1024 positions or more. 36 shapes, time by three over that by two wavefronts with shared stages:
//     documents of 256 to 900 0.75 to 0.86, whole rows 0.67 to 0.87, 100 to 200 0.88 to 1.02, 16 to 64 from 548 row blocks on
//     0.89 to 1.00 (one call of 66 1.05), 60 to 120 0.93 to 1.04 up to 671 row blocks and 0.94 to 1.08 from 672 on. Us,
//     documents of 32 to 64, 100 to 200, 400 to 500, whole rows: [1, 4608, 4/4], 576 row blocks, 9.6 -> 8.8, 10.6 -> 9.6,
//     15.8 -> 13.0, 68 -> 51; [1, 6144, 4/4], 768, 10.7 -> 9.7, 11.1 -> 11.1, 16.9 -> 13.9, 91 -> 71.
//     The lower line: up to 512 the workgroups of four wavefronts are all there at once. From 516 to 536 documents of 16 to 64
//     lose 2 to 10 % in 25 of 34 calls of one to twelve heads ([1, 8320, 2/2], 520, 8.4 -> 9.1), at 540 and 544 2 to 7 % in 5
//     of 14, from 548 to 556 in none of 12; longer ones gain throughout ([1, 4224, 4/4], 528, 400 to 500, 16.1 -> 13.2;
//     [1, 4352, 4/4], 544, whole rows 64.6 -> 48.7). The upper one: heads in no multiple of four put keys of all heads on
//     every XCD. From 600 on documents of 60 to 120 lose 2 to 24 % in 49 of 55 calls of one to ten heads, of 100 to 200 2 to 16 % in
//     46 ([1, 3840, 5/5], 600, 10.2 -> 10.9, 11.1 -> 12.4; [1, 10368, 2/2], 648, 10.4 -> 11.3, 11.1 -> 11.7); up to 592 the first 0
//     to 4 % in 7, the second none. Shared keys lose with short documents (they are staged for every head: [1, 2304, 8/2], 576,
//     8.2 -> 8.7, though 14.7 -> 12.0 and 37 -> 29 with longer ones), and so does a second round (832, 10.8 -> 12.5).
//   head dimension 64: sharing by two wins up to between 6144 (62 against 77 us with a long document) and 8192 (52 against 47).
//   head dimension 128: sharing by two wins below 2048 (42 against 55 us at 1920) where rows see many keys; short documents lose
//     there (four heads that share keys, 1536 row blocks, documents of up to 128 13.9 / 10.2 by whole row blocks, [3, 4608, 4/4]
//     images 58 / 93), and the host does not know them. A little over one round of tiles in long rows of image blocks (a call with
//     ends says so) still waits for the longest rows' chains: by two / a tile each [1, 4224, 16/4] 57 / 70 us, [1, 17152, 4/1] 86 /
//     109, [2, 5504, 6/2] 77 / 91, [4, 4992, 4/4] 111 / 99; 19 shapes 1.08 times. Shorter rows lose ([1, 3200, 24/8] 58 / 50), and
//     so do more blocks ([3, 4864, 8/2] alike, [1, 30208, 4/4] 160 / 130) and whole rows without ends ([1, 9216, 8/2] 203 / 177).
//     Rows of up to 20 key tiles: pieces of 64 keys on their own ([8, 768, 24/4], documents of 61 to 122, 29 us, by query tiles
//     32; whole rows of 1280, [4, 1280, 32/8], 65 / 63). Longer ones: a query tile per workgroup of four wavefronts
//     (attn_fwd_tile_kernel). Workgroups of eight that walk the metadata's bins are ahead only where the tiles of four heads that
//     share keys fill the places exactly twice, so that nothing evens out what the pairs leave: 3841 to 4096 row blocks, us
//     so / a tile each, [1, 8192, 16/4] whole rows 242 / 249, [1, 16384, 8/2] 466 / 484, [2, 4096, 16/4] 128.7 / 132.3, [6, 2688,
//     8/1] images 92 / 95; [1, 6144, 32/8], 6144 blocks, whole rows 287 / 277.
template <int D>
static int dispatch_fwd(hipStream_t stream, const AttnParams& p) {
  const long blocks = (long)p.B * p.Hq * (p.S / 32);
  if constexpr (D == 64) {
    if (blocks <= 512) return p.S >= 1024 ? launch_fwd_shares<D, 8>(stream, p) : launch_fwd_shares<D, 4>(stream, p);
    if (blocks <= 768 && p.S >= 512) return launch_fwd_shares<D, 4>(stream, p);
    if (blocks < 7168) return launch_fwd_split<D, 4, 2, 1, 1>(stream, p);
    return launch_fwd_split<D, 4, 1, 1, 2>(stream, p);
  } else {
    if (blocks <= 256 && p.S >= 1024) return launch_fwd_shares<D, 8>(stream, p);
    if (blocks <= 512) return launch_fwd_shares<D, 4>(stream, p);
    if (p.Hq == p.Hkv && p.S >= 1024 && blocks > 536 && blocks <= (p.Hq % 4 == 0 ? 768 : 592))
      return launch_fwd_shares<D, 3>(stream, p);
    if (blocks < 2048 || (p.end && blocks < 2560 && p.S >= 56 * kKeyTile)) return launch_fwd_split<D, 4, 2, 1, 1>(stream, p);
    if (p.S <= 20 * kKeyTile) return launch_fwd_split<D, 4, 1, 2, 1>(stream, p);
    switch (heads_per_group(p.Hq, p.Hkv)) {
      case 4: return blocks > 3840 && blocks <= 4096 ? launch_fwd<D, 4>(stream, p) : launch_fwd_tile<4>(stream, p);
      case 2: return launch_fwd_tile<2>(stream, p);
      default: return launch_fwd_tile<1>(stream, p);
    }
  }
}

// Workgroups of the persistent dQ kernels: two or three per compute unit, the same number for every (head slice, KV head) group.
// Where the groups do not share the places evenly some have a member less at first, and members behind the places go on with
// those groups' tiles as places come free: up to twice as many, 64 or 96 a group at most. (That many for any number of groups were
// up to 6144 workgroups, which still had to be started when all tiles were taken. dQ, us, so / now: [3, 5632, 24/8 heads of 64],
// documents of 64 to 300, 79 / 72; [3, 1536, 64/64 of 64] whole rows 129 / 123; from stored blocks [2, 4096, 36/12 of 128], 16 to
// 100, 42 / 36, [8, 768, 64/8 of 64] 53 / 48. No further members at all: [4, 5760, 48/16 of 128] 337 / 349, with them 344.)
static int dq_grid(const AttnParams& p, int hs, int per_unit = 2) {
  const int groups = ((p.Hq / p.Hkv) / hs) * p.kvh_count;
  const int places = per_unit * kBins * 8, members = (places + groups - 1) / groups;
  return groups * (places % groups == 0 ? members : std::min(2 * members, std::max(members, per_unit * kBins)));
}

template <int D, int HS, int PER_UNIT>
static int launch_dq(hipStream_t stream, const AttnParams& p) {
  const size_t smem = 2 * KvStage<D>::kBytes;
  CT_ENSURE_LDS("ct_attn_bwd", (&attn_dq_kernel<D, HS, PER_UNIT>), smem);
  LaunchScope scope2("attn_dq_kernel", stream);
  hipLaunchKernelGGL((attn_dq_kernel<D, HS, PER_UNIT>), dim3(dq_grid(p, HS, PER_UNIT)), dim3(256), smem, stream, p);
  return scope2.done();
}
// (where the line lies: attn_dq_kernel)
template <int D, int HS>
static int launch_dq(hipStream_t stream, const AttnParams& p) {
  if constexpr (D == 64)
    if ((long)p.B * p.Hq * (p.S / 32) >= 12288) return launch_dq<D, HS, 3>(stream, p);
  return launch_dq<D, HS, 2>(stream, p);
}

// `reduce`: the launch also adds the chunks of split key tiles. Beside a workgroup per tile (KS > 1) by 128 workgroups of eight
// wavefronts: there can be many more pieces than these 1024 wavefronts (17408 at [1, 3072, 32/32 of 128]), which then take several
// each. A pass, us, with the sums in a launch of their own / by 128 / by 256: [2, 1024, 8/8 of 64], whole rows,
// 40.7 / 38.0 / 37.5; [1, 2304, 6/1 of 64], documents of 256 to 900, 39.6 / 38.7 / 34.3; [1, 2688, 16/16 of 64], whole rows,
// 91.6 / 87.4 / 88.0; [4, 1792, 16/8 of 64] 153.5 / 152.6 / 148.5; [1, 3072, 32/32 of 128] 311 / 306 / 301; [2, 1536, 8/2 of
// 128], documents of 32 to 128, 46.1 / 41.4 / 42.3. Over 33 calls of 64 to 8192 row blocks 0.88 to 1.01 of their own launch.
// Behind workgroups that pull tiles (KS = 1) by 512, as many wavefronts as a launch of their own has (attn_dq_blocks_kernel).
template <int D, int HS, int KS>
static int launch_dq_blocks(hipStream_t stream, const AttnParams& p, bool reduce) {
  const size_t smem = DsStage<D, KS>::kTotalBytes;
  CT_ENSURE_LDS("ct_attn_bwd", (&attn_dq_blocks_kernel<D, HS, KS>), smem);
  const int groups = p.Hq / p.Hkv / HS * p.kvh_count;
  const int grid = KS == 1 ? dq_grid(p, HS) : groups * p.B * bin_tiles_per_row(p.S / 32, kDqbWaves / KS / HS);
  const int reduce_groups = !reduce ? 0 : KS > 1 ? 128 : 512;
  LaunchScope scope("attn_dq_blocks_kernel", stream);
  hipLaunchKernelGGL((attn_dq_blocks_kernel<D, HS, KS>), dim3(grid + reduce_groups), dim3(kDqbWaves * 64), smem, stream, p, reduce_groups);
  return scope.done();
}

// By the row blocks of the launch (32 query rows of one head). The kernel lives on the bytes it has in flight: in
// large launches 16 wavefronts per compute unit and work pulling, in small ones the walk of the longest row is the
// time, two key blocks in flight, and sharing it shortens the walk and puts more of it in flight. Measured
// (us, one wavefront per row block / two / four), rows with documents of up to the row or images of 1056:
//   136 row blocks, D = 128: 47 / 24 / 17      432, D = 64: 43 / 23 / 15       608, D = 64: 26 / 14 / 10
//   1088, D = 64: 43 / 23 / 21 and 22 / 12 / 13, short documents 16 / 7 / 12   1776, D = 128: 44 / 35 / 42
//   2880, D = 64: 34 / 19 / 29                 8928, D = 64: 248 / 248
//   3744, D = 128: 124 / 102 / 127, but 2.5 us slower by two with short documents (a compute unit holds one of its
//   workgroups, of the others two); 7680: 201 / 227
// Stored blocks that were chosen for their small number (most_stored_blocks) are shared by two up to 10240 row blocks, as the
// walks are short: the backward, D = 64, by one / two, [11, 384, 64/16], 8448, documents of 16 to 64, 92 / 84 us, of 128 to 192
// 97 / 92; [22, 768, 16/4], 8448, 256 to 384, 109 / 110; [32, 768, 16/4], 12288, 145 / 149, 16 to 64 97 / 98; 24576: 193 / 208.
template <int D>
static int dispatch_dq_blocks(hipStream_t stream, const AttnParams& p, bool reduce) {
  const long blocks = (long)p.B * p.kvh_count * (p.Hq / p.Hkv) * (p.S / 32);
  const int hs = heads_per_group(p.Hq, p.Hkv);
  if (blocks <= 768) return hs == 1 ? launch_dq_blocks<D, 1, 4>(stream, p, reduce) : launch_dq_blocks<D, 2, 4>(stream, p, reduce);
  if (blocks <= (D == 128 ? 3072 : p.ds_most_blocks ? 10240 : 8192))
    return hs == 4   ? launch_dq_blocks<D, 4, 2>(stream, p, reduce)
           : hs == 2 ? launch_dq_blocks<D, 2, 2>(stream, p, reduce)
                     : launch_dq_blocks<D, 1, 2>(stream, p, reduce);
  return hs == 4   ? launch_dq_blocks<D, 4, 1>(stream, p, reduce)
         : hs == 2 ? launch_dq_blocks<D, 2, 1>(stream, p, reduce)
                   : launch_dq_blocks<D, 1, 1>(stream, p, reduce);
}

// Which dK/dV kernel runs for head dimension 128 when the caller leaves the choice open: the wide one's streams, of one wavefront
// per SIMD, are ahead only where nearly every step of a long walk is all-allowed (whole rows) and every compute unit has key tiles
// to the end. Recomputing backward of [B, S, heads / KV heads], us, narrow / wide, 50 calls:
//   whole rows, (key tile, KV head) pairs beyond the places: [1, 16384, 32/8] 6779 / 6548, [2, 16384, 16/4] 6710 / 6475; where KV
//     heads have no group or one of eight 3275 / 3294 ([1, 16384, 16/16]), 53789 / 54627 ([1, 32768, 64/8])
//   up to 320 pairs: [1, 16384, 2/1] 677 / 724, 8/2 1844 / 1950, [1, 32768, 8/1] 7256 / 7698, [1, 20480, 6/2] 2118 / 2220
//   packed documents, of 512 to the whole row: 0.80 to 0.98 of the wide one's time ([1, 32768, 64/8] 25121 / 26978), of 512 to 2048
//     0.82 to 0.94, of 64 to 300 0.78 to 0.87, image blocks 0.84 to 0.94.
// The documents are the device's to see: long rows launch both kernels, the wide one first, and count the visited blocks.
constexpr int kWideDkvFromSeq = 16384;
static int wide_least_blocks(const AttnParams& p) {
  const long nrb = p.S / 32, pairs = (long)p.B * (p.S / kDkvKeys) * p.Hkv;
  const long whole = p.B * (nrb * (nrb + 1) / 2);
  return pairs <= kDkvSlots ? INT_MAX : (int)std::min(whole * 9 / 10, (long)INT_MAX);
}

// One pass of the dK/dV kernel over the KV heads p.kvh_base ... (all of them unless dS is stored).
template <int D>
static int launch_dkv(hipStream_t stream, const AttnParams& p, bool wide) {
  const size_t smem = QdoStage<D>::kTotalBytes;
  const int grid = p.dkv_max_entries * p.kvh_count;  // entries beyond the list's length exit at once
  if constexpr (D == 128) {
    if (wide) {
      CT_ENSURE_LDS("ct_attn_bwd", &attn_dkv_wide_kernel, DkvWideLds::kTotalBytes);
      LaunchScope scope("attn_dkv_wide_kernel", stream);
      hipLaunchKernelGGL(attn_dkv_wide_kernel, dim3(grid), dim3(128), DkvWideLds::kTotalBytes, stream, p);
      if (p.dkv_by_blocks) {  // (timed with it: one of the two exits at once)
        CT_ENSURE_LDS("ct_attn_bwd", (&attn_dkv_kernel<D, false>), smem);
        hipLaunchKernelGGL((attn_dkv_kernel<D, false>), dim3(grid), dim3(256), smem, stream, p);
      }
      return scope.done();
    }
  }
  LaunchScope scope3("attn_dkv_kernel", stream);
  if constexpr (D == 64) {
    if (p.dq_rides) {
      const int hs = heads_per_group(p.Hq, p.Hkv);
      const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), std::max(smem, (size_t)2 * KvStage<D>::kBytes), stream, p);
      };
      if (hs == 4) launch(attn_dkv_then_dq_kernel<4>);
      else if (hs == 2) launch(attn_dkv_then_dq_kernel<2>);
      else launch(attn_dkv_then_dq_kernel<1>);
      return scope3.done();
    }
    if (p.ds_most_blocks) {
      CT_ENSURE_LDS("ct_attn_bwd", &attn_dkv_choice_kernel<D>, smem);
      hipLaunchKernelGGL(attn_dkv_choice_kernel<D>, dim3(grid), dim3(256), smem, stream, p);
      return scope3.done();
    }
  }
  if (p.ds) {
    CT_ENSURE_LDS("ct_attn_bwd", (&attn_dkv_kernel<D, true>), smem);
    hipLaunchKernelGGL((attn_dkv_kernel<D, true>), dim3(grid), dim3(256), smem, stream, p);
  } else {
    CT_ENSURE_LDS("ct_attn_bwd", (&attn_dkv_kernel<D, false>), smem);
    hipLaunchKernelGGL((attn_dkv_kernel<D, false>), dim3(grid), dim3(256), smem, stream, p);
  }
  return scope3.done();
}

template <int D>
static int launch_dkv_reduce(hipStream_t stream, const AttnParams& p) {
  LaunchScope scope9("attn_dkv_reduce_kernel", stream);
  hipLaunchKernelGGL((attn_dkv_reduce_kernel<D>), dim3(kReduceGroups), dim3(256), 0, stream, p);
  return scope9.done();
}

// The delta pass on its own: delta in row order (b, s, h).
template <int D>
static int launch_delta(hipStream_t stream, const bf16* out, const bf16* dout, float* delta, long rows) {
  // 16 workgroups per compute unit, each walking 1024-chunk tiles with a grid stride
  const long tiles = (rows * (D / 8) + 1023) / 1024;
  const dim3 grid((unsigned)(tiles < 4096 ? tiles : 4096));
  LaunchScope scope4("attn_delta_kernel", stream);
  hipLaunchKernelGGL((attn_delta_kernel<D>), grid, dim3(256), 0, stream, out, dout, delta, rows);
  return scope4.done();
}

template <int D>
static int launch_schedule(hipStream_t stream, const AttnParams& p, int kvh_side_by_side) {
  LaunchScope scope7("attn_dkv_schedule_kernel", stream);
  hipLaunchKernelGGL(attn_dkv_schedule_kernel<D>, dim3(1), dim3(1024), 0, stream, p, kvh_side_by_side);
  return scope7.done();
}

// dQ per query tile: evaluates S and dP itself and computes delta and -lse / scale for its rows on the way.
template <int D>
static int dispatch_dq(hipStream_t stream, const AttnParams& p) {
  switch (heads_per_group(p.Hq, p.Hkv)) {
    case 4: return launch_dq<D, 4>(stream, p);
    case 2: return launch_dq<D, 2>(stream, p);
    default: return launch_dq<D, 1>(stream, p);
  }
}

// Recompute form: the work list; dQ; dK/dV per key tile; the sum of split chunks.
template <int D>
static int dispatch_bwd_recompute(hipStream_t stream, const AttnParams& p, bool wide, bool list_kept) {
  int rc = list_kept ? 0 : launch_schedule<D>(stream, p, p.Hkv);
  if (rc) return rc;
  rc = dispatch_dq<D>(stream, p);
  if (rc) return rc;
  rc = launch_dkv<D>(stream, p, wide);
  if (rc) return rc;
  return launch_dkv_reduce<D>(stream, p);
}

// The most dS blocks per query head with which dQ comes from stored blocks, 0 where the form is settled (see kDqRecomputes).
// Recomputing is ahead from about 42000 blocks (of all heads) and 2.3 per row block on, sooner per row block the larger the launch.
// At 8192 row blocks stored ones are what a call gets (their bits are part of what callers hold this size to), below the recomputing
// tiles ride with dK/dV (dq_rides); under 3072 row blocks those end unevenly: backward kernels, us, stored / so, [2, 2816, 16/16 of
// 64], documents of 1408 to 2816, 110 / 124, [2, 3200, 12/4], images, 107 / 116, though [2, 4096, 10/2], whole rows, 227 / 190.
// 36 drawn calls from 3072 on 0.985 to 1.43, 1.048 in the geometric mean.
// Backward beyond 8192, in us, stored / this / recomputing (head dimension 64):
//   [3, 1536, 64/16]  9216 row blocks, documents of 16 to 64 93 / 90 / 103, of 512 to 768 165 / 152 / 149, whole rows 323 / 260 / 257
//   [4, 4096, 64/16] 32768, 16 to 64 261 / 263 / 269, 1365 to 2048 875 / 690 / 702, whole rows 2475 / 1826 / 1826
//   [12, 4096, 8/8] 12288, whole rows 1028 / 732 / 736, image blocks 596 / 445 / 473
// Over 70 shapes of 8200 to 61000 row blocks: short documents 0.93 to 1.02 of the stored form's time, long ones 0.71 to 0.9.
constexpr long kStoredRowBlocks = 8192;
static int most_stored_blocks(const AttnParams& p, int head_dim) {
  const long rows = (long)p.B * p.Hq * (p.S / 32);
  if (head_dim != 64 || rows < 3072 || rows == kStoredRowBlocks) return 0;
  return (int)((42000 + 2.3 * rows) / p.Hq);
}

// Stored-dS form: row statistics and the work list; then per pass of KV heads the dK/dV kernel, which
// leaves its dS blocks in the region, and dQ as a product over those blocks; the sum of split chunks. With p.ds_most_blocks the
// recomputing dQ stands between the first two, and forms the statistics, where the header asks for it, or rides with the second.
template <int D>
static int dispatch_bwd_blocks(hipStream_t stream, AttnParams p, int kvh_per_pass, bool wide, bool list_kept) {
  const long tiles = (long)p.B * p.Hq * (p.S / (D == 128 ? 64 : 128));
  const unsigned stats_groups = (unsigned)(tiles < 8192 ? tiles : 8192);
  int rc;
  if (list_kept) {
    LaunchScope scope("attn_bwd_stats_kernel", stream);
    hipLaunchKernelGGL((attn_bwd_stats_kernel<D>), dim3(stats_groups), dim3(256), 0, stream, p, exponent_scale(p.scale));
    rc = scope.done();
  } else {
    LaunchScope scope("attn_dkv_schedule_kernel", stream);  // (the list and the statistics)
    hipLaunchKernelGGL((attn_bwd_setup_kernel<D>), dim3(1 + (stats_groups + 3) / 4), dim3(1024), 0, stream, p, kvh_per_pass,
                       exponent_scale(p.scale));
    rc = scope.done();
  }
  if (rc) return rc;
  if constexpr (D == 64) {
    if (p.ds_most_blocks && !p.dq_rides) rc = dispatch_dq<D>(stream, p);
    if (rc) return rc;
  }
  for (int base = 0; base < p.Hkv; base += kvh_per_pass) {
    p.kvh_base = base;
    p.kvh_count = min(kvh_per_pass, p.Hkv - base);
    rc = launch_dkv<D>(stream, p, wide);
    if (rc) return rc;
    // (with the last pass all chunks are there)
    rc = dispatch_dq_blocks<D>(stream, p, base + p.kvh_count == p.Hkv);
    if (rc) return rc;
  }
  return CT_OK;
}

}  // namespace ct

using namespace ct;

extern "C" size_t ct_attn_meta_bytes(int32_t batch, int32_t seq) {
  if (batch <= 0 || seq <= 0) return 0;
  return meta_total_ints(batch, seq / 32) * sizeof(int32_t);
}

static bool bwd_shape_ok(int32_t batch, int32_t seq, int32_t q_heads, int32_t kv_heads, int32_t head_dim) {
  return batch > 0 && seq > 0 && q_heads > 0 && kv_heads > 0 && head_dim > 0 && seq % kDkvKeys == 0 &&
         q_heads % kv_heads == 0;
}

extern "C" size_t ct_attn_bwd_workspace_bytes(int32_t batch, int32_t seq, int32_t q_heads,
                                             int32_t kv_heads, int32_t head_dim) {
  if (!bwd_shape_ok(batch, seq, q_heads, kv_heads, head_dim)) return 0;
  return bwd_plan(batch, seq, q_heads, kv_heads, head_dim, false, 0, false).total;
}

extern "C" size_t ct_attn_bwd_workspace_bytes_from_ds(int32_t batch, int32_t seq, int32_t q_heads,
                                                     int32_t kv_heads, int32_t head_dim,
                                                     int32_t has_attention_end) {
  if (!bwd_shape_ok(batch, seq, q_heads, kv_heads, head_dim)) return 0;
  const BwdPlan plan = bwd_plan(batch, seq, q_heads, kv_heads, head_dim, has_attention_end != 0, 0, true);
  return plan.spill ? plan.total : 0;
}

static_assert(kFusedRows / 32 <= kPrepareLdsRowBlocks, "the fused form keeps the row's records in LDS");

static int32_t prepare_on(const char* fn, void* stream, const int32_t* segment_ids, const int32_t* attention_end,
                          int32_t batch, int32_t seq, int32_t* tile_meta, SummaryOut queries, SummaryOut keys) {
  CT_REQUIRE(segment_ids && tile_meta, "%s: null pointer", fn);
  int rc = validate_shape(fn, batch, seq, 1, 1, 128);
  if (rc) return rc;
  const int nrb = seq / 32;
  // working arrays: LDS when they fit, else the scratch region after the table
  int* scratch = tile_meta + meta_table_ints(batch, nrb);
  int* prepare_scratch = nullptr;
  if (!prepare_fits_lds(nrb)) {
    prepare_scratch = scratch;
    scratch += (size_t)batch * 3 * nrb;
  }
  int* bins_scratch = bins_fit_lds(batch, nrb) ? nullptr : scratch;
  hipStream_t st = (hipStream_t)stream;
  if ((long)batch * seq <= kOneLaunchPositions && seq <= kFusedRows) {
    const int tiles = batch * bin_tiles_per_row(nrb, 2);
    const size_t smem = ((size_t)5 * batch * nrb + (3 * tiles > nrb ? 3 * tiles : nrb)) * sizeof(int);
    LaunchScope scope("attn_prepare_kernel", st);
    hipLaunchKernelGGL(attn_prepare_kernel, dim3(3 + 6 * batch + (nrb + 63) / 64 * batch), dim3(1024), smem, st, tile_meta, batch, seq,
                       queries, keys, segment_ids, attention_end, tile_meta + (size_t)batch * nrb * kMetaW);
    return scope.done();
  }
  const bool fused = seq <= kFusedRows;
  if (!fused) {
    LaunchScope scope5("attn_blocks_kernel", st);
    hipLaunchKernelGGL(attn_blocks_kernel, dim3((seq + 1023) / 1024, batch), dim3(1024), 0, st, segment_ids, attention_end, seq,
                       tile_meta);
    if ((rc = scope5.done())) return rc;
  }
  CT_ENSURE_LDS(fn, &attn_ranges_kernel<true>, kPrepareLdsRowBlocks * 3 * 4);
  LaunchScope scope6("attn_ranges_kernel", st);
  hipLaunchKernelGGL((prepare_scratch ? attn_ranges_kernel<false> : attn_ranges_kernel<true>), dim3((nrb + 63) / 64, batch),
                     dim3(1024), prepare_scratch ? 0 : (size_t)nrb * 3 * sizeof(int), st, tile_meta, seq, queries, keys, fused ? segment_ids : nullptr, attention_end);
  if ((rc = scope6.done())) return rc;
  const size_t bins_smem = bins_scratch ? 0 : (size_t)3 * batch * bin_tiles_per_row(nrb, 2) * sizeof(int);
  const size_t row_smem = prepare_scratch ? 0 : (size_t)nrb * sizeof(int);
  CT_ENSURE_LDS(fn, &attn_schedules_kernel, kBinsLdsInts * 4);
  LaunchScope scope8("attn_schedules_kernel", st);
  hipLaunchKernelGGL(attn_schedules_kernel, dim3(3 + 6 * batch), dim3(1024), bins_smem > row_smem ? bins_smem : row_smem, st,
                     tile_meta, batch, seq, tile_meta + (size_t)batch * nrb * kMetaW, prepare_scratch, bins_scratch);
  return scope8.done();
}

extern "C" int32_t ct_attn_prepare(void* stream, const int32_t* segment_ids,
                                   const int32_t* attention_end, int32_t batch, int32_t seq,
                                   int32_t* tile_meta) {
  return prepare_on("ct_attn_prepare", stream, segment_ids, attention_end, batch, seq, tile_meta, SummaryOut{}, SummaryOut{});
}

extern "C" int32_t ct_attn_prepare_summaries(void* stream, const int32_t* segment_ids, const int32_t* attention_end,
                                             int32_t batch, int32_t seq, int32_t* tile_meta, int32_t block_q,
                                             int32_t* q_summary, int32_t block_kv, int32_t* kv_summary) {
  CT_REQUIRE(q_summary && kv_summary, "ct_attn_prepare_summaries: null pointer");
  CT_REQUIRE(block_q > 0 && block_q % 32 == 0 && block_kv > 0 && block_kv % 32 == 0 && seq > 0 && seq % block_q == 0 &&
                 seq % block_kv == 0,
             "ct_attn_prepare_summaries: blocks %d and %d must be multiples of 32 that divide the sequence %d", block_q,
             block_kv, seq);
  return prepare_on("ct_attn_prepare_summaries", stream, segment_ids, attention_end, batch, seq, tile_meta,
                    SummaryOut{q_summary, block_q, attention_end ? 3 : 2}, SummaryOut{kv_summary, block_kv, 2});
}

extern "C" int32_t ct_attn_block_summary(void* stream, const int32_t* segment_ids,
                                         const int32_t* attention_end, int32_t batch, int32_t seq,
                                         int32_t block, int32_t* out) {
  CT_REQUIRE(segment_ids && out, "ct_attn_block_summary: null pointer");
  CT_REQUIRE(batch > 0 && seq > 0 && block > 0, "ct_attn_block_summary: dimensions must be positive");
  CT_REQUIRE(seq % block == 0, "ct_attn_block_summary: sequence %d not divisible by block %d", seq,
             block);
  const int nblocks = batch * (seq / block);
  LaunchScope scope6("attn_block_summary_kernel", (hipStream_t)stream);
  hipLaunchKernelGGL(attn_block_summary_kernel, dim3((nblocks + 3) / 4), dim3(256), 0,
                     (hipStream_t)stream, segment_ids, attention_end, block, nblocks,
                     attention_end ? 3 : 2, out);
  return scope6.done();
}

extern "C" int32_t ct_attn_fwd(void* stream, const ct_attn_fwd_args* a) {
  CT_REQUIRE(a, "ct_attn_fwd: null args");
  CT_REQUIRE(a->q && a->k && a->v && a->segment_ids && a->tile_meta && a->out && a->lse,
             "ct_attn_fwd: null pointer");
  int rc = validate_shape("ct_attn_fwd", a->batch, a->seq, a->q_heads, a->kv_heads, a->head_dim);
  if (rc) return rc;
  CT_REQUIRE(a->scale == a->scale && a->scale - a->scale == 0.f, "ct_attn_fwd: scale must be finite");
  CT_REQUIRE(aligned16({a->q, a->k, a->v, a->segment_ids, a->attention_end, a->tile_meta, a->out, a->lse}),
             "ct_attn_fwd: every device pointer must be 16-byte aligned");
  AttnParams p = {};
  p.q = reinterpret_cast<const bf16*>(a->q);
  p.k = reinterpret_cast<const bf16*>(a->k);
  p.v = reinterpret_cast<const bf16*>(a->v);
  p.seg = a->segment_ids;
  p.end = a->attention_end;
  p.meta = a->tile_meta;
  p.sched = a->tile_meta + (size_t)a->batch * (a->seq / 32) * kMetaW;
  p.out = reinterpret_cast<bf16*>(a->out);
  p.lse = a->lse;
  p.B = a->batch;
  p.S = a->seq;
  p.Hq = a->q_heads;
  p.Hkv = a->kv_heads;
  p.scale = round_to_bf16(a->scale);
  return a->head_dim == 128 ? dispatch_fwd<128>((hipStream_t)stream, p)
                            : dispatch_fwd<64>((hipStream_t)stream, p);
}

extern "C" int32_t ct_attn_delta(void* stream, const uint16_t* out, const uint16_t* dout,
                                 float* delta, int64_t rows, int32_t head_dim) {
  CT_REQUIRE(out && dout && delta, "ct_attn_delta: null pointer");
  CT_REQUIRE(rows > 0, "ct_attn_delta: rows must be positive");
  CT_REQUIRE(aligned16({out, dout, delta}), "ct_attn_delta: every device pointer must be 16-byte aligned");
  if (head_dim != 64 && head_dim != 128)
    return fail(CT_UNSUPPORTED, "ct_attn_delta: head_dim must be 64 or 128, got %d", head_dim);
  const bf16* o = reinterpret_cast<const bf16*>(out);
  const bf16* g = reinterpret_cast<const bf16*>(dout);
  return head_dim == 128 ? launch_delta<128>((hipStream_t)stream, o, g, delta, (long)rows)
                         : launch_delta<64>((hipStream_t)stream, o, g, delta, (long)rows);
}

extern "C" int32_t ct_attn_bwd(void* stream, const ct_attn_bwd_args* a) {
  CT_REQUIRE(a, "ct_attn_bwd: null args");
  CT_REQUIRE(a->q && a->k && a->v && a->segment_ids && a->tile_meta && a->out && a->lse &&
                 a->dout && a->dq && a->dk && a->dv && a->delta && a->workspace,
             "ct_attn_bwd: null pointer");
  int rc = validate_shape("ct_attn_bwd", a->batch, a->seq, a->q_heads, a->kv_heads, a->head_dim);
  if (rc) return rc;
  CT_REQUIRE(a->scale == a->scale && a->scale - a->scale == 0.f, "ct_attn_bwd: scale must be finite");
  CT_REQUIRE(aligned16({a->q, a->k, a->v, a->segment_ids, a->attention_end, a->tile_meta, a->out, a->lse,
                        a->dout, a->dq, a->dk, a->dv, a->delta, a->workspace}),
             "ct_attn_bwd: every device pointer must be 16-byte aligned");
  AttnParams p = {};
  p.q = reinterpret_cast<const bf16*>(a->q);
  p.k = reinterpret_cast<const bf16*>(a->k);
  p.v = reinterpret_cast<const bf16*>(a->v);
  p.seg = a->segment_ids;
  p.end = a->attention_end;
  p.meta = a->tile_meta;
  p.sched = a->tile_meta + (size_t)a->batch * (a->seq / 32) * kMetaW;
  p.out = const_cast<bf16*>(reinterpret_cast<const bf16*>(a->out));
  p.lse = const_cast<float*>(a->lse);
  p.dout = reinterpret_cast<const bf16*>(a->dout);
  p.delta = a->delta;
  p.dq = reinterpret_cast<bf16*>(a->dq);
  p.dk = reinterpret_cast<bf16*>(a->dk);
  p.dv = reinterpret_cast<bf16*>(a->dv);
  p.B = a->batch;
  p.S = a->seq;
  p.Hq = a->q_heads;
  p.Hkv = a->kv_heads;
  p.scale = round_to_bf16(a->scale);
  const int kernel_choice = a->variant & 0xf, path_choice = a->variant & 0xf0;
  const bool list_kept = (a->variant & CT_ATTN_BWD_WORK_LIST_KEPT) != 0;
  CT_REQUIRE((a->variant & ~(0xff | CT_ATTN_BWD_WORK_LIST_KEPT)) == 0 && kernel_choice <= CT_ATTN_BWD_DKV_WIDE &&
                 (path_choice == 0 || path_choice == CT_ATTN_BWD_DQ_RECOMPUTE || path_choice == CT_ATTN_BWD_DQ_FROM_DS),
             "ct_attn_bwd: unknown variant 0x%x", a->variant);
  // The wide dK/dV kernel does not store dS: asking for it settles the dQ form as well.
  const bool wide_forced = kernel_choice == CT_ATTN_BWD_DKV_WIDE && a->head_dim == 128;
  CT_REQUIRE(!(wide_forced && path_choice == CT_ATTN_BWD_DQ_FROM_DS),
             "ct_attn_bwd: the wide dK/dV kernel has no stored-dS form");
  // Left to the library (no form asked for), the stored-dS form runs where it costs nothing the caller has
  // not offered: rows of up to CT_ATTN_FROM_DS_UP_TO_SEQ positions (measured: beside the flag in ct_hotpath.h), the
  // narrow dK/dV kernel, and a workspace that holds the dS blocks of all KV heads at once.
  bool allow_blocks = path_choice == CT_ATTN_BWD_DQ_FROM_DS;
  if (path_choice == 0 && !wide_forced && a->seq <= CT_ATTN_FROM_DS_UP_TO_SEQ) {
    const BwdPlan offered = bwd_plan(a->batch, a->seq, a->q_heads, a->kv_heads, a->head_dim,
                                     a->attention_end != nullptr, a->workspace_bytes, true);
    allow_blocks = offered.spill && offered.kvh_per_pass == a->kv_heads && a->workspace_bytes >= offered.total;
  }
  const BwdPlan plan = bwd_plan(a->batch, a->seq, a->q_heads, a->kv_heads, a->head_dim,
                                a->attention_end != nullptr, a->workspace_bytes, allow_blocks);
  if (a->workspace_bytes < plan.total)
    return fail(CT_WORKSPACE_TOO_SMALL, "ct_attn_bwd: workspace %zu < %zu bytes", a->workspace_bytes,
                plan.total);
  if (path_choice == CT_ATTN_BWD_DQ_FROM_DS && !plan.spill)
    return fail(CT_WORKSPACE_TOO_SMALL,
                "ct_attn_bwd: the stored-dS form needs %zu bytes of workspace for one KV head, got %zu",
                plan.L.total + ds_bytes_per_kv_head(a->batch, a->seq, a->q_heads, a->kv_heads,
                                                    a->attention_end != nullptr),
                a->workspace_bytes);
  const DkvLayout& L = plan.L;
  char* ws = static_cast<char*>(a->workspace);
  p.dkv_header = reinterpret_cast<int*>(ws + L.header);
  p.dq_counters = p.dkv_header + 64;
  p.dkv_entries = reinterpret_cast<int2*>(ws + L.entries);
  p.dkv_partials = reinterpret_cast<float*>(ws + L.partials);
  p.lse2 = reinterpret_cast<float*>(ws + L.lse2);
  p.dkv_max_entries = L.max_entries;
  p.dkv_max_partials = L.max_partials;
  p.kvh_base = 0;
  p.kvh_count = a->kv_heads;
  if (a->head_dim == 128 && a->seq >= kWideDkvFromSeq) p.wide_least_blocks = wide_least_blocks(p);
  hipStream_t s = (hipStream_t)stream;
  if (plan.spill) {
    p.ds = ws + plan.ds;
    p.ds_row_blocks = plan.row_blocks;
    if (path_choice == 0) p.ds_most_blocks = most_stored_blocks(p, a->head_dim);
    p.dq_rides = p.ds_most_blocks && (long)p.B * p.Hq * (p.S / 32) < kStoredRowBlocks;
    // (every group of heads needs a workgroup of that launch)
    if (p.dq_rides && p.Hq / heads_per_group(p.Hq, p.Hkv) > p.dkv_max_entries * p.Hkv) p.ds_most_blocks = p.dq_rides = 0;
    return a->head_dim == 128 ? dispatch_bwd_blocks<128>(s, p, plan.kvh_per_pass, false, list_kept)
                              : dispatch_bwd_blocks<64>(s, p, plan.kvh_per_pass, false, list_kept);
  }
  p.dkv_by_blocks = kernel_choice == 0 && p.wide_least_blocks;
  const bool wide = wide_forced || p.dkv_by_blocks;
  return a->head_dim == 128 ? dispatch_bwd_recompute<128>(s, p, wide, list_kept)
                            : dispatch_bwd_recompute<64>(s, p, wide, list_kept);
}
