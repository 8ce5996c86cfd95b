// Projection-fused cut cross-entropy for gfx950: kernels and C ABI.
//
// Forward (logits never reach memory):
//   prepare  stable list of active rows (weight != 0) -> gather indices; an aligned copy of a head whose rows are not
//   stats    persistent GEMM workgroups: logits^T tile = head_tile^T hidden_tile^T,
//            folded on the fly into per-row running (max, sum exp, target logit)
//            for one (vocab chunk, row block) unit at a time
//   merge    combine the vocab chunks per row -> lse, weighted loss, block sums; the last workgroup adds
//            those in a fixed order -> nll_sum, weight_sum
// Backward:
//   prepare  the same list, the constants of its rows, the active rows packed; the head as above
//   dlogits  G = w * dy * (exp(logits - lse) - onehot), rounded to bf16, written
//            vocabulary-major to a workspace slab G^T [vocab slab, rows]
//   dhidden  dHidden = G head^T
//   dhead    dHead   = hidden^T G
// The reference recomputes the logits in both backward kernels
// (src/kernels/cut_cross_entropy.py:258, :383); here G is formed once and shared,
// which keeps the reference's rounding points (G is cast to bf16 before both
// products, :272, :396). Its logits come either from a second GEMM (4 GEMMs
// instead of the reference's 5) or, when the caller lends the forward a cache,
// from the f32 logits the forward left there (3 GEMMs, the algorithmic count).
// The cache is vocabulary-major [vocab, rows] like G^T: in the transposed tile
// the GEMMs produce, the lanes of a wavefront run along the rows, so both are
// written with contiguous stores.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "ct_error.h"
#include "ct_gemm.hip.h"

namespace ct {

constexpr int kBK = kGemmBK;
constexpr int kComputeUnits = 256;    // of an MI355X; sizes of work units are chosen by it
constexpr float kNegInfF = -__builtin_inff();

struct CutceHeader {
  int n_act;
  int counter;
  // per-XCD work counters: set 0 statistics kernel / hidden gradient, set 1 head gradient,
  // set 2 the dlogits kernel that recomputes the projection
  int xcd_counter[3][8];
  int pad[6];
};

// Clears counter sets 0 and 1 (called by workgroup 0 of a kernel that runs before their users).
CT_DEVICE void reset_unit_counters(CutceHeader* header) {
  if (threadIdx.x < 16) (&header->xcd_counter[0][0])[threadIdx.x] = 0;
}
// Clears counter set 2.
CT_DEVICE void reset_dlogits_counters(CutceHeader* header) {
  if (threadIdx.x < 8) header->xcd_counter[2][threadIdx.x] = 0;
}

// Work order of the persistent GEMM kernels. A unit is a pair (a, b) of operand tile indices,
// a < a_count, b < b_count; every unit is one 256 x 256 GEMM tile (or a run of them) that
// reads tile a of one operand and tile b of the other. A workgroup asks for its next unit ahead (request), so that
// the counter's answer travels behind an epilogue, or in the projection kernels behind the last GEMM of the unit.
//
// Plain order, up to kPlainRounds units per workgroup: the grid is walked with a as the slow index, the
// first unit of a workgroup is its own number, the others come from one counter. Within a round
// every XCD gets an eighth of the units, consecutive ones, which share operands; a last round that fills only part of the
// device likewise (one round of the statistics kernel, every unit on the next XCD / consecutive ones, us: 380 x 17624,
// d = 1664, 414 small tiles 47.8 / 37.0; 385 x 3120, d = 7296, 100 small ones 72.9 / 68.4; 335 x 28712, d = 2432, 226 large ones
// 66.3 / 61.8). A list of units of two lengths (`mixed`) that is over in less than a round is dealt to the XCDs one by
// one: the long ones would meet on some of them (both gradients of 4000 x 1900, d = 1024: 39.8 / 43.9). (Short problems have no use for the orders
// below: counters of XCDs that own nothing, indices that fall outside ragged grids and rounds of
// asking the other XCDs cost 10-20 us a launch.)
//
// Each XCD has its own L2, so in large problems the workgroups of one XCD should work at the same time
// on units that share operands. Blocks: the (a, b) grid is walked in blocks of kA x kB = 32 units (the
// 32 compute units of an XCD: 4 + 8 operand tiles feed 32 GEMM tiles), the sequence of blocks is cut
// into 8 equal ranges, and an XCD takes the units of its range through its own counter. Indices that
// fall outside the grid (ragged edges) are skipped. An XCD that runs dry helps the next one.
//
// Sweep (the two projection kernels, a = vocabulary chunk, b = row block): XCD x owns the
// row blocks x, x + 8, ... and walks (a, its row blocks) with a as the slow index, so all eight
// XCDs are on the same few vocabulary chunks at the same time. The head is the large operand
// (1 GB against 0.1 GB of hidden rows): with every XCD on the same chunk it leaves HBM about once
// per pass, and the other XCDs find it in the memory-side cache; in block mode each XCD streams
// its own range of the vocabulary and the head is read from HBM once per 8 row blocks.
constexpr int kPlainRounds = 8;
struct UnitQueue {
  static constexpr int kA = 4, kB = 8, kXcds = 8;
  enum Order { kPlain, kBlocks, kSweep };
  int* counters;
  int a_count, b_count, total, b_groups, padded_total, per_xcd, my_xcd;
  int helping;  // how many XCDs further the counter in use belongs to
  Order order;
  bool requested, started, mixed;
  int pending;  // of thread 0: the counter's answer
  CT_DEVICE void init(int* counters_, int a_count_, int b_count_, Order large, bool mixed_ = false) {
    counters = counters_;
    a_count = a_count_;
    b_count = b_count_;
    total = a_count * b_count;
    order = total <= kPlainRounds * (int)gridDim.x ? kPlain : large;
    mixed = mixed_;
    b_groups = (b_count + kB - 1) / kB;
    padded_total = ((a_count + kA - 1) / kA) * b_groups * kA * kB;
    per_xcd = (padded_total + kXcds - 1) / kXcds;
    unsigned xcc_id;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc_id));
    my_xcd = (int)(xcc_id & 7u);
    helping = 0;
    requested = started = false;
  }
  CT_DEVICE void request() {
    // (an address that is not known to be uniform: for a uniform one the compiler adds once per wavefront and
    // distributes the answer, for which it waits on the spot)
    int which = order == kPlain ? 0 : (my_xcd + helping) % kXcds;
    asm volatile("" : "+v"(which));
    if (threadIdx.x == 0) pending = atomicAdd(counters + which, 1);
    requested = true;
  }
  // The answer, for all threads of the workgroup (contains barriers).
  CT_DEVICE int receive(int* lds_slot) {
    if (!requested) request();
    requested = false;
    if (threadIdx.x == 0) *lds_slot = pending;
    __syncthreads();
    const int answer = uniform(*lds_slot);  // scalar from here on: unit indices feed scalar address arithmetic
    __syncthreads();
    return answer;
  }
  CT_DEVICE int next_plain(int* lds_slot) {
    const int n = gridDim.x;
    const int i = started ? n + receive(lds_slot) : (int)blockIdx.x;
    started = true;
    const int round = i / n * n, in = min(n, total - round), at = i - round;
    if (at >= in || (in < n && round == 0 && mixed)) return i;
    return round + at % kXcds * (in / kXcds) + min(at % kXcds, in % kXcds) + at / kXcds;
  }
  // Called by all threads of the workgroup (contains barriers); false when nothing is left.
  CT_DEVICE bool next(int& a, int& b, int* lds_slot) {
    if (order == kPlain) {
      const int i = next_plain(lds_slot);
      a = i / b_count;
      b = i % b_count;
      return i < total;
    }
    while (helping < kXcds) {
      const int x = (my_xcd + helping) % kXcds;
      if (order == kSweep) {
        const int mine = x < b_count ? (b_count - x + kXcds - 1) / kXcds : 0;  // row blocks of XCD x
        const int local = receive(lds_slot);
        if (local < a_count * mine) {
          a = local / mine;
          b = x + kXcds * (local % mine);
          return true;
        }
      } else {
        const int local = receive(lds_slot);
        const int index = x * per_xcd + local;
        if (local < per_xcd && index < padded_total) {
          const int in_block = index % (kA * kB), block = index / (kA * kB);
          a = (block / b_groups) * kA + in_block / kB;
          b = (block % b_groups) * kB + in_block % kB;
          if (a < a_count && b < b_count) return true;
          continue;
        }
      }
      ++helping;
    }
    return false;
  }
};

// The head as the GEMM kernels read it: column v of row n at base[n * ld + v - col0]. Either the
// caller's tensor (ld = V) or, where its rows are not 16-byte aligned (V % 8 != 0) and it is not read in place
// (forward_in_place, backward_in_place), an aligned copy of the columns col0 .. in the workspace ("panel", HeadCopy), padded with
// zero columns to whole tiles.
// An aligned head whose vocabulary is no multiple of 128 has the columns from the last such multiple
// on a second time in `tail` [d][128], padded with zeros, for the contraction over the vocabulary; an unaligned
// one that is read in place the columns from the last multiple of 256 on in `tail` [d][256], for that and for the
// projections' last tile: nothing past the end of a row is read from the caller's tensor.
struct HeadView {
  const bf16* base;
  const bf16* tail;
  long ld;
  int col0;
  int tail_first, tail_cols;  // vocabulary id of the tail's first column, and its row length
  bool padded;
};

struct CutceParams {
  const bf16* hidden;
  HeadView head;
  const int* targets;
  const float* weights;
  int N, d, V, n_pad;
  int compact;
  int* idx;            // [n_pad] row of each slot
  int* slot_target;    // [n_pad] forward: target of each slot, -1 for a row without weight
  int* block_active;   // [n_pad / 256] forward: whether a block of slots has a row with weight
  CutceHeader* header;
  bool hidden_aligned;

  // columns of the head that a tile at v0 may read, relative to the view
  CT_DEVICE const int* gather() const { return compact ? idx : nullptr; }  // (slots are rows otherwise)
  CT_DEVICE int head_cols(int v0) const { return head.padded ? v0 - head.col0 + kGemmTile : V - head.col0; }
};

// ---------------------------------------------------------------------------
// index: stable compaction of active rows (and, for the backward, their constants)
// ---------------------------------------------------------------------------
// Forward. Workgroup b places the rows 1024 b .. 1024 b + 1023; it counts the active rows in front of them
// by itself (N floats, from L2 for all but the first reader), so no workgroup waits for another: one
// pass of latency instead of one per 1024 rows (27 -> 5 us at N = 16384).
CT_DEVICE void list_rows(const CutceParams& p, int block, int blocks) {
  __shared__ int wave_total[16], wave_first[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int begin = block * 1024, i = begin + tid;
  const bool last = block == blocks - 1;
  if (last) {
    reset_unit_counters(p.header);
    reset_dlogits_counters(p.header);
  }
  const float w = i < p.N ? p.weights[i] : 0.f;
  const bool active = w != 0.f;
  int slot = i, total = p.N, filler = 0;
  bool placed = i < p.N;
  if (p.compact) {
    int count = 0, first = p.N;  // active rows of this wavefront's share in front of `begin`
    for (int base = 0; base < begin; base += 1024) {
      const unsigned long long ballot = __ballot(p.weights[base + tid] != 0.f);
      if (ballot) first = min(first, base + wave * 64 + __ffsll(ballot) - 1);
      count += __popcll(ballot);
    }
    const unsigned long long ballot = __ballot(active);
    if (ballot) first = min(first, begin + wave * 64 + __ffsll(ballot) - 1);
    if (lane == 0) {
      wave_total[wave] = count;
      wave_first[wave] = first;
    }
    __syncthreads();
    int before = 0;
    filler = p.N;
    for (int k = 0; k < 16; ++k) {
      before += wave_total[k];
      filler = min(filler, wave_first[k]);
    }
    filler = filler < p.N ? filler : 0;  // keeps gathers past the end on a live row
    __syncthreads();
    if (lane == 0) wave_total[wave] = __popcll(ballot);
    __syncthreads();
    total = before;
    for (int k = 0; k < 16; ++k) {
      if (k < wave) before += wave_total[k];
      total += wave_total[k];
    }
    slot = before + __popcll(ballot & ((1ull << lane) - 1ull));
    placed = active;
  }
  const unsigned long long ballot = __ballot(active);
  __syncthreads();
  if (lane == 0) wave_first[wave] = ballot != 0;
  __syncthreads();
  const int* any = wave_first + (wave & ~3);
  if (lane == 0 && (wave & 3) == 0 && i < p.n_pad)
    p.block_active[i / kGemmTile] = p.compact || any[0] || any[1] || any[2] || any[3];
  if (placed) {
    p.idx[slot] = i;
    p.slot_target[slot] = active ? p.targets[i] : -1;
  }
  if (!last) return;
  for (int k = total + tid; k < p.n_pad; k += 1024) {
    p.idx[k] = filler;
    p.slot_target[k] = -1;
  }
  if (tid == 0) {
    p.header->n_act = total;
    p.header->counter = 0;
  }
}

// Per-slot constants of the backward: (w dy, lse log2 e, target), zeros / -1 past the active rows.
struct CutceRowParams {
  float* fac;
  float* lse2;
  int* tgt;
};
// What the row work of the backward reads and writes beside the list.
struct CutceRowWork {
  const float* lse;
  const float* dy;
  CutceRowParams rp;
  bf16* packed;   // [n_pad][d], or null
  bf16* dhidden;
};

// Backward. A workgroup of 16 wavefronts places rows_per_group(N, d) rows and does their row work, one or
// several per row: packed[slot] = hidden[row], and zeros for the dHidden rows of ignored tokens. (The head gradient
// contracts over slots; with the rows packed its operand tiles are plain strided copies instead of a gather at
// every step. The slots past the active rows up to the next multiple of 256 hold zeros; their G^T entries
// are zero or not read.) Every workgroup counts all weights by itself, from L2, and no workgroup waits for
// another; a wavefront's first row is on its way meanwhile. The list and the row work in two launches took
// 4.5 + 4.8 us at N = 380, d = 1664, now 5.8, and 9.2 + 40 at N = 16384, d = 4096. One round everywhere makes
// the counting the longer part (69 us there).
// Few long rows are shared by several wavefronts each, for more workgroups: a compute unit moves about 50 GB/s (a wavefront
// per row / four, us: 64 rows, d = 6400 13.4 / 8.4, 250 10.0 / 7.4, 1000 12.1 / 9.8; d = 2048 6.8 / 6.1, 6.0 / 6.1,
// 6.8 / 6.9, and 1024 and less 0.2 longer, d = 1280 to 1792 0.8 less to 0.7 longer; two, 2000 rows: d = 2048 9.0 / 8.2, 6400
// 13.3 / 12.5).
constexpr int kMostRowRounds = 64;
__host__ __device__ inline int row_rounds(int rows) { return min((rows + 4095) / 4096, kMostRowRounds); }
__host__ __device__ inline int row_waves(int rows, int d) { return d < 2048 || rows > 2048 ? 1 : rows > 1024 ? 2 : 4; }
__host__ __device__ inline int rows_per_group(int rows, int d) { return 16 * row_rounds(rows) / row_waves(rows, d); }
constexpr int kAhead = 8;         // chunks of a row per lane that are read while the weights are counted
CT_DEVICE void list_and_pack_rows(const CutceParams& p, const CutceRowWork& work, int block, int blocks) {
  __shared__ int wave_before[16], wave_total[16], wave_first[16], group_count[16], slot_of[16 * kMostRowRounds];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rounds = row_rounds(p.N), waves = row_waves(p.N, p.d), rows = rows_per_group(p.N, p.d);
  const int begin = block * rows, row_chunks = p.d / 8;
  // the wavefront's row of a round, and its chunks of the row: lane0 + stride k
  const int group_row = wave / waves, lane0 = wave % waves * 64 + lane, stride = 64 * waves;
  if (block == 0) {
    reset_unit_counters(p.header);
    reset_dlogits_counters(p.header);
  }
  const bool ahead = work.packed && p.hidden_aligned;
  u32x4 chunk[kAhead];
  const auto row_chunk = [&](int row, int c) {
    return reinterpret_cast<const u32x4*>(p.hidden + (size_t)min(row, p.N - 1) * p.d)[min(c, row_chunks - 1)];
  };
  if (ahead) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) chunk[k] = row_chunk(begin + group_row, lane0 + stride * k);
  }
  int before = begin, total = p.N, filler = 0;
  if (p.compact) {
    int count_before = 0, count = 0, first = p.N;
#pragma unroll 4
    for (int base = 0; base < p.N; base += 1024) {
      const int i = base + tid;
      const unsigned long long ballot = __ballot(i < p.N && p.weights[i] != 0.f);
      const int row0 = base + wave * 64;  // of this wavefront's 64 rows
      count += __popcll(ballot);
      const int in_front = min(max(begin - row0, 0), 64);
      count_before += __popcll(in_front == 64 ? ballot : ballot & ((1ull << in_front) - 1ull));
      if (ballot) first = min(first, row0 + __ffsll(ballot) - 1);
    }
    if (lane == 0) {
      wave_before[wave] = count_before;
      wave_total[wave] = count;
      wave_first[wave] = first;
    }
    __syncthreads();
    before = total = 0;
    filler = p.N;
    for (int k = 0; k < 16; ++k) {
      before += wave_before[k];
      total += wave_total[k];
      filler = min(filler, wave_first[k]);
    }
    filler = filler < p.N ? filler : 0;  // keeps gathers past the end on a live row
  }
  // the list: wavefront g places the g-th 64 rows of the workgroup
  const int local = wave * 64 + lane, i = begin + local;
  const bool mine = local < rows && i < p.N;
  const float w = mine ? p.weights[i] : 0.f;
  const unsigned long long ballot = __ballot(w != 0.f);
  if (lane == 0) group_count[wave] = __popcll(ballot);
  __syncthreads();
  for (int g = 0; g < wave; ++g) before += p.compact ? group_count[g] : 0;
  const bool placed = mine && (!p.compact || w != 0.f);
  const int slot = p.compact ? before + __popcll(ballot & ((1ull << lane) - 1ull)) : i;
  if (local < rows) slot_of[local] = placed ? slot : -1;
  if (placed) {
    p.idx[slot] = i;
    work.rp.fac[slot] = w != 0.f ? w * work.dy[0] : 0.f;
    work.rp.lse2[slot] = w != 0.f ? work.lse[i] * kLog2e : __builtin_inff();
    work.rp.tgt[slot] = w != 0.f ? p.targets[i] : -1;
  }
  if (block == 0 && tid == 0) {
    p.header->n_act = total;
    p.header->counter = 0;
  }
  // the slots past the active rows, shared by the workgroups
  for (int k = total + block * 1024 + tid; k < p.n_pad; k += blocks * 1024) {
    p.idx[k] = filler;
    work.rp.fac[k] = 0.f;
    work.rp.lse2[k] = __builtin_inff();
    work.rp.tgt[k] = -1;
  }
  __syncthreads();
  for (int round = 0; round < rounds; ++round) {
    const int in_group = 16 / waves * round + group_row, row = begin + in_group;
    if (row >= p.N) break;
    if (p.weights[row] == 0.f) {
      u32x4* dst = reinterpret_cast<u32x4*>(work.dhidden + (size_t)row * p.d);
      for (int c = lane0; c < row_chunks; c += stride) dst[c] = u32x4{0u, 0u, 0u, 0u};
    }
    const int slot = uniform(slot_of[in_group]);
    if (!work.packed || slot < 0) continue;
    u32x4* dst = reinterpret_cast<u32x4*>(work.packed + (size_t)slot * p.d);
    if (ahead) {
      if (round != 0) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) chunk[k] = row_chunk(row, lane0 + stride * k);
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        if (lane0 + stride * k < row_chunks) dst[lane0 + stride * k] = chunk[k];
#pragma unroll 4
      for (int c = lane0 + stride * kAhead; c < row_chunks; c += stride) dst[c] = row_chunk(row, c);
    } else {
      const bf16* from = p.hidden + (size_t)row * p.d;
      for (int c = lane0; c < p.d; c += stride) reinterpret_cast<bf16*>(dst)[c] = from[c];
    }
  }
  if (work.packed) {
    const int end = (total + kGemmTile - 1) / kGemmTile * kGemmTile;
    for (int k = total + block * 16 + wave; k < end; k += blocks * 16) {
      u32x4* dst = reinterpret_cast<u32x4*>(work.packed + (size_t)k * p.d);
      for (int c = lane; c < p.d / 8; c += 64) dst[c] = u32x4{0u, 0u, 0u, 0u};
    }
  }
}

// ---------------------------------------------------------------------------
// The head as the GEMM loop can copy it
// ---------------------------------------------------------------------------
// With V % 8 != 0 the rows of the head start at addresses that are multiples of 2 bytes only, and
// the asynchronous copies of the GEMM loop move aligned 16-byte chunks. One pass over the head
// (2 bytes read and written per element) makes them usable: the guarded loop that loads such
// rows element by element runs at 20-90 TFLOP/s against the pipelined one's 600-1300. The pass needs nothing
// that the row lists make, so it shares their launch.
struct HeadCopy {
  const bf16* head;
  bf16* panel;  // `cols` (a multiple of 256) columns from col0 on, zero-padded, or null
  bf16* tail;   // HeadView::tail, or null
  int col0, cols;
  int tail_first, tail_cols;
};
constexpr int kPanelRows = 4, kPanelColumns = 2048;  // of 256 threads
__host__ __device__ inline int head_copy_blocks(const HeadCopy& copy, int d) {
  if (copy.panel) return (copy.cols + kPanelColumns - 1) / kPanelColumns * (d / (4 * kPanelRows));
  return copy.tail ? (d * (copy.tail_cols / 8) + 1023) / 1024 : 0;
}
CT_DEVICE void copy_head(const HeadCopy& copy, int V, int d, int block) {
  const int tid = threadIdx.x;
  if (copy.panel) {
    const int col_blocks = (copy.cols + kPanelColumns - 1) / kPanelColumns;
    const int c = ((block % col_blocks) * 256 + (tid & 255)) * 8, row0 = ((block / col_blocks) * 4 + (tid >> 8)) * kPanelRows;
    if (c >= copy.cols) return;
    const int left = V - (copy.col0 + c);
    const bf16* src = copy.head + (size_t)row0 * V + copy.col0 + c;
    bf16* dst = copy.panel + (size_t)row0 * copy.cols + c;
    bf16x8 v[kPanelRows];
    if (left >= 8) {
#pragma unroll
      for (int r = 0; r < kPanelRows; ++r) __builtin_memcpy(&v[r], src + (size_t)r * V, 16);
    } else {
      for (int r = 0; r < kPanelRows; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[r][e] = e < left ? src[(size_t)r * V + e] : (bf16)0.f;
    }
#pragma unroll
    for (int r = 0; r < kPanelRows; ++r) store_global16(dst + (size_t)r * copy.cols, as_u32x4(v[r]));
  } else {
    const int chunks = copy.tail_cols / 8, index = block * 1024 + tid, row = index / chunks, c = index % chunks * 8;
    if (row >= d) return;
    const bf16* src = copy.head + (size_t)row * V + copy.tail_first + c;
    const int left = V - (copy.tail_first + c);
    bf16x8 chunk;
    if (left >= 8) {
      __builtin_memcpy(&chunk, src, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) chunk[e] = e < left ? src[e] : (bf16)0.f;
    }
    store_global16(copy.tail + (size_t)row * copy.tail_cols + c, as_u32x4(chunk));
  }
}

// The first list_blocks workgroups make the row list, the others copy the head. A launch that only copies (a
// further part of the vocabulary) has list_blocks = 0; `reset`: the statistics kernel that follows starts from
// fresh work counters.
template <bool BACKWARD>
__global__ __launch_bounds__(1024) void cutce_prepare_kernel(CutceParams p, CutceRowWork work, HeadCopy copy, int list_blocks,
                                                             bool reset) {
  const int block = blockIdx.x;
  if (block >= list_blocks) {
    if (reset && block == 0) reset_unit_counters(p.header);
    copy_head(copy, p.V, p.d, block - list_blocks);
  } else if constexpr (BACKWARD) {
    list_and_pack_rows(p, work, block, list_blocks);
  } else {
    list_rows(p, block, list_blocks);
  }
}

// ---------------------------------------------------------------------------
// stats
// ---------------------------------------------------------------------------
CT_DEVICE void merge_stats(float& m, float& s, float m_o, float s_o) {
  const float m_new = fmaxf(m, m_o);
  const float m_use = (m_new == kNegInfF) ? 0.f : m_new;
  s = s * exp2_fast(m - m_use) + s_o * exp2_fast(m_o - m_use);
  m = m_new;
}

// The head's tile of a projection, vocabulary ids v0 ..
template <GemmLoads LOADS, int NB>
CT_DEVICE void head_tile(McLoader<NB>& A, const CutceParams& p, int v0) {
  if constexpr (LOADS == GemmLoads::kThroughRegisters) {
    const bool inside = v0 + GemmShape<NB>::kTile <= p.V;
    const int first = inside ? v0 : v0 - p.head.tail_first;
    A.init(inside ? p.head.base : p.head.tail, inside ? p.head.ld : p.head.tail_cols, first, first + GemmShape<NB>::kTile, p.d);
  } else {
    A.init(p.head.base, p.head.ld, v0 - p.head.col0, p.head_cols(v0), p.d);
  }
}

// Bound by the matrix pipe at long contractions; at short ones by what lies between two products, for the large tile
// has its compute unit to itself. In clocks a tile, 4096 x 32000 at d = 256: product 10.1 k (8.2 k of MFMAs), first
// copies of the next tile 2.5 k (96 KB at 64 bytes a clock), epilogue 8.5 k, end of a unit 2.4 k; the copies'
// latency, the cleared accumulators and a second reading of them in the epilogue took 116 us to 104 there, 67 to 65
// at 900 x 32003, d = 1024, 175 to 162 at 1845 x 67203, d = 512. (Small tiles on two workgroups per compute unit, whose epilogues could
// fall behind each other's products: 152, 81 and 196, bound by the bytes that reach LDS.)
template <int NB, bool CACHE, GemmLoads LOADS, int RING = 4>
__global__ __launch_bounds__(256, (GemmShape<NB, RING>::kGroups)) void cutce_stats_kernel(CutceParams p, float* part, int chunk0, int chunks,
                                                                    int tiles_per_chunk, float* cache) {
  constexpr int kTile = GemmShape<NB>::kTile, kWave = GemmShape<NB>::kWave;
  extern __shared__ __align__(16) char smem_raw[];
  const lds_addr smem = lds_address_of(smem_raw);
  __shared__ int unit_s;
  __shared__ float exch[2 * kWave * 3];  // [2 wn][kWave rows][3]
  const int tid = threadIdx.x, l = tid & 63, j = l & 31, half = l >> 5, w = tid >> 6;
  const int wm = (w >> 1) * kWave, wn = (w & 1) * kWave;
  const int vocab_tiles = (p.V + kTile - 1) / kTile;
  const int n_act = p.header->n_act;

  // units: (vocabulary chunk, row block); row blocks in which no row carries weight are passed over
  const int active_blocks = (n_act + kTile - 1) / kTile;
  UnitQueue units;
  units.init(p.header->xcd_counter[0], chunks, active_blocks, UnitQueue::kSweep);
  const auto next_unit = [&](int& chunk, int& rb) {
    while (units.next(chunk, rb, &unit_s))
      if (p.compact || p.block_active[rb * kTile / kGemmTile]) return true;
    return false;
  };
  int chunk, rb;
  bool more = next_unit(chunk, rb);
  McLoader<NB> A;
  GemmB<NB, LOADS> B;
  GemmTiles<NB, LOADS, CACHE, RING> gemm;
  // Rows are interleaved in the tile (KcLoader): column block nb of lane j is row slot
  // n0 + wn + NB j + nb, so a lane owns NB consecutive slots.
  typedef int LaneInts __attribute__((ext_vector_type(NB)));
  LaneInts next_tgt;
  // The loaders of a tile and the copies of its first steps. What a new unit loads for its epilogues is waited for
  // here, where nothing else is in flight: a wait behind the epilogue's stores would be one for them too.
  const auto begin_tile = [&](int vt, bool new_unit) {
    if (new_unit) {
      next_tgt = *reinterpret_cast<const LaneInts*>(p.slot_target + rb * kTile + wn + NB * j);
      B.init(p.hidden, p.d, p.gather(), rb * kTile, n_act, p.d, true);
      asm volatile("" : "+v"(next_tgt));
    }
    head_tile<LOADS>(A, p, vt * kTile);
    gemm.begin(A, B, smem);
  };
  if (more) begin_tile((chunk0 + chunk) * tiles_per_chunk, true);
  while (more) {
    const int n0 = rb * kTile, part_row = chunk0 + chunk;
    const LaneInts tgt = next_tgt;
    float m2[NB], sum[NB], tl[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      m2[nb] = kNegInfF;
      sum[nb] = 0.f;
      tl[nb] = 0.f;
    }

    const int vt_end = min((part_row + 1) * tiles_per_chunk, vocab_tiles);
    for (int vt = part_row * tiles_per_chunk; vt < vt_end; ++vt) {
      const int v0 = vt * kTile;
      const bool last = vt + 1 == vt_end;
      if (last) units.request();
      GemmAcc<NB> acc;
      gemm.run(A, B, p.d, smem, acc);
      if (last) more = next_unit(chunk, rb);
      if (more) begin_tile(last ? (chunk0 + chunk) * tiles_per_chunk : vt + 1, last);

      const int vbase = v0 + wm + 4 * half;  // vocab id of (i, r) = vbase + 32 i + 8 (r/4) + r%4
      const bool ragged = v0 + kTile > p.V;
      if constexpr (CACHE) {
        // cache^T[v][slot]: a lane stores its NB consecutive slots with one access, 32
        // lanes = NB * 128 contiguous bytes. Address = wave-uniform tile origin + uniform row offset +
        // a 32-bit lane offset, so the stores need no per-store vector address arithmetic.
        float* origin = cache + (size_t)(v0 + uniform(wm)) * p.n_pad + n0 + uniform(wn);
        const unsigned lane_off = (unsigned)(4 * half * p.n_pad + NB * j) * 4u;  // bytes
        TileRows rows(origin, p.n_pad * 4);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) gemm.store(rows, lane_off, r, acc.lane(i, r));
      }
      // A column block's 16 NB elements are read once. (The limit is opaque: comparison masks kept for the next
      // block do not fit and spill, and so is every 16 elements' result, or their use is put off past a branch.)
      const auto fold = [&](auto ragged_tile) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          float x[16 * NB];
          int limit = p.V - vbase;
          if (ragged_tile.value) asm volatile("" : "+v"(limit));
          float tmax = kNegInfF;
#pragma unroll
          for (int i = 0; i < NB; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              float& e = x[16 * i + r];
              e = acc.value(i, nb, r);
              if (ragged_tile.value && 32 * i + acc_row(r, 0) >= limit) e = kNegInfF;
            }
#pragma unroll
            for (int r = 0; r < 16; r += 2) tmax = fmaxf(fmaxf(x[16 * i + r], x[16 * i + r + 1]), tmax);  // (v_max3)
            asm volatile("" : "+v"(tmax));
          }
          const int rel = tgt[nb] - (v0 + wm);
          if (__any(rel >= 0 && rel < kWave)) {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
#pragma unroll
              for (int r = 0; r < 16; ++r) tl[nb] += vbase + 32 * i + acc_row(r, 0) == tgt[nb] ? x[16 * i + r] : 0.f;
              asm volatile("" : "+v"(tl[nb]));
            }
          }
          const float m_new = fmaxf(m2[nb], tmax * kLog2e);
          const float m_use = (m_new == kNegInfF) ? 0.f : m_new;
          float add = 0.f;
#pragma unroll
          for (int i = 0; i < NB; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) add += exp2_fast(x[16 * i + r] * kLog2e - m_use);
            asm volatile("" : "+v"(add));
          }
          sum[nb] = sum[nb] * exp2_fast(m2[nb] - m_use) + add;
          m2[nb] = m_new;
        }
      };
      if (ragged) fold(std::true_type{});
      else fold(std::false_type{});
    }

    // lanes l and l^32 hold the same rows; then the two wavefronts with equal wn.
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      merge_stats(m2[nb], sum[nb], xor32(m2[nb]), xor32(sum[nb]));
      tl[nb] += xor32(tl[nb]);
    }
    if (wm != 0 && half == 0) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        float* e = exch + ((w & 1) * kWave + 32 * nb + j) * 3;
        e[0] = m2[nb];
        e[1] = sum[nb];
        e[2] = tl[nb];
      }
    }
    __syncthreads();
    if (wm == 0 && half == 0) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float* e = exch + ((w & 1) * kWave + 32 * nb + j) * 3;
        merge_stats(m2[nb], sum[nb], e[0], e[1]);
        tl[nb] += e[2];
        float* out = part + ((size_t)part_row * p.n_pad + n0 + wn + NB * j + nb) * 3;
        out[0] = m2[nb];
        out[1] = sum[nb];
        out[2] = tl[nb];
      }
    }
    // (the next unit's GEMM lies between these LDS reads and its writes)
  }
}

// ---------------------------------------------------------------------------
// merge
// ---------------------------------------------------------------------------
// A workgroup merges the per-chunk partials of kMergeSlots row slots: PARTS threads per slot each walk every
// PARTS-th vocabulary chunk, then the parts are combined in a fixed order: the two of a wavefront, then the
// wavefronts. The pass is bound by the latency of those walks, so long ones are shared by 32 threads, short
// ones by 8 (us with 8 / 32: 60 rows x 1002 chunks 12.7 / 9.2, 128 x 300 8.4 / 5.9, 384 x 167 5.7 / 5.4; 64 x 5
// 4.2 / 4.7, 4000 x 15 5.5 / 6.0).
constexpr int kMergeSlots = 32, kShortMerge = 64;
template <int PARTS>
__global__ __launch_bounds__(kMergeSlots * PARTS) void cutce_merge_kernel(CutceParams p, const float* part, int chunks,
                                                                          float* lse_out, double* block_sums,
                                                                          float* nll_sum, float* weight_sum_out) {
  constexpr int kWaves = kMergeSlots * PARTS / 64;
  __shared__ float exch[kWaves][kMergeSlots][3];
  __shared__ double red[2][64];
  __shared__ bool last_s;
  const int tid = threadIdx.x, lane_slot = tid % kMergeSlots, piece = tid / kMergeSlots;
  const int slot = blockIdx.x * kMergeSlots + lane_slot;
  const int n_act = p.header->n_act;
  double loss = 0.0, wsum = 0.0;
  if (piece == 0 && slot < p.N) {
    const float wi = p.weights[slot];
    wsum = (double)wi;
    if (wi == 0.f) lse_out[slot] = 0.f;
  }
  int row = 0;
  float wr = 0.f;
  if (slot < n_act) {
    row = p.idx[slot];
    wr = p.weights[row];
  }
  float m = kNegInfF, s = 0.f, t = 0.f;
  if (slot < n_act) {  // (not by wr, which is still on its way; a row without weight is not stored below)
#pragma unroll 4
    for (int c = piece; c < chunks; c += PARTS) {  // (several chunks' loads in flight)
      const float* e = part + ((size_t)c * p.n_pad + slot) * 3;
      merge_stats(m, s, e[0], e[1]);
      t += e[2];
    }
  }
  merge_stats(m, s, xor32(m), xor32(s));
  t += xor32(t);
  if (piece % 2 == 0) {
    exch[piece / 2][lane_slot][0] = m;
    exch[piece / 2][lane_slot][1] = s;
    exch[piece / 2][lane_slot][2] = t;
  }
  __syncthreads();
  if (piece == 0) {
    if (wr != 0.f) {
      for (int k = 1; k < kWaves; ++k) {
        merge_stats(m, s, exch[k][lane_slot][0], exch[k][lane_slot][1]);
        t += exch[k][lane_slot][2];
      }
      const float lse = (__log2f(s) + m) * kLn2;
      lse_out[row] = lse;
      loss = (double)wr * ((double)lse - (double)t);
    }
    red[0][lane_slot] = loss;
    red[1][lane_slot] = wsum;
  }
  __syncthreads();
  // The sums of the workgroups are added by the one that ends last, in a fixed order: lane l adds the blocks l,
  // l + 64, ..., then the lanes are added. They pass through memory by device-scope atomics only, and the answer of
  // the exchange is what the counter's increment waits for (a fence would write back the L2).
  const auto bits = reinterpret_cast<unsigned long long*>(block_sums);
  if (tid < 2) {
    double sum = 0.0;
    for (int k = 0; k < kMergeSlots; ++k) sum += red[tid][k];  // fixed order
    unsigned long long was = __hip_atomic_exchange(bits + 2 * blockIdx.x + tid, __builtin_bit_cast(unsigned long long, sum),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(was) : : "memory");
    // (both lanes' exchanges have been answered: they are one instruction of the wavefront)
    if (tid == 0)
      last_s = __hip_atomic_fetch_add(&p.header->counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
  }
  __syncthreads();
  if (!last_s || tid >= 64) return;
  double total[2] = {0.0, 0.0};
  for (int b = tid; b < (int)gridDim.x; b += 64)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      total[k] += __builtin_bit_cast(double, __hip_atomic_load(bits + 2 * b + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  red[0][tid] = total[0];
  red[1][tid] = total[1];
  __builtin_amdgcn_wave_barrier();
  if (tid >= 2) return;
  double sum = 0.0;
  for (int k = 0; k < 64; ++k) sum += red[tid][k];
  *(tid ? weight_sum_out : nll_sum) = (float)sum;
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
CT_DEVICE float dlogit(float logit, float fac, float lse2, int tgt, int v) {
  return fac * (exp2_fast(logit * kLog2e - lse2) - (v == tgt ? 1.f : 0.f));
}

// G^T[v - slab0][slot], logits recomputed (transposed tile as in the statistics kernel: rows =
// vocabulary, lanes = row slots). Persistent like the statistics kernel and with its unit order:
// a unit is tiles_per_chunk vocabulary tiles of the slab times one block of 256 active rows.
template <int NB, GemmLoads LOADS, int RING = 4>
__global__ __launch_bounds__(256, (GemmShape<NB, RING>::kGroups)) void cutce_dlogits_kernel(CutceParams p, CutceRowParams rp,
                                                                      int slab0, int slab_tiles, int tiles_per_chunk,
                                                                      bf16* G) {
  constexpr int kTile = GemmShape<NB>::kTile, kWave = GemmShape<NB>::kWave;
  typedef float LaneFloats __attribute__((ext_vector_type(NB)));
  typedef int LaneInts __attribute__((ext_vector_type(NB)));
  extern __shared__ __align__(16) char smem_raw[];
  const lds_addr smem = lds_address_of(smem_raw);
  __shared__ int unit_s;
  const int tid = threadIdx.x, l = tid & 63, j = l & 31, half = l >> 5, w = tid >> 6;
  const int wm = (w >> 1) * kWave, wn = (w & 1) * kWave;
  const int n_act = p.header->n_act;
  // the two GEMM kernels that follow start from fresh work counters
  if (blockIdx.x == 0) reset_unit_counters(p.header);
  const int active_blocks = (n_act + kTile - 1) / kTile;  // G^T columns past them are never used
  const int chunks = (slab_tiles + tiles_per_chunk - 1) / tiles_per_chunk;
  UnitQueue units;
  units.init(p.header->xcd_counter[2], chunks, active_blocks, UnitQueue::kSweep);
  int chunk, rb;
  bool more = units.next(chunk, rb, &unit_s);
  McLoader<NB> A;
  GemmB<NB, LOADS> B;
  GemmTiles<NB, LOADS, true, RING> gemm;
  // Rows are interleaved in the tile (KcLoader): column block nb of lane j is row slot
  // n0 + wn + NB j + nb, so a lane owns NB consecutive slots of G^T and stores them together.
  LaneFloats next_fac, next_lse2;
  LaneInts next_tgt;
  const auto begin_tile = [&](int vt, bool new_unit) {  // as in the statistics kernel
    const int v0 = slab0 + vt * kTile;
    if (new_unit) {
      const int slot = rb * kTile + wn + NB * j;
      next_fac = *reinterpret_cast<const LaneFloats*>(rp.fac + slot);
      next_lse2 = *reinterpret_cast<const LaneFloats*>(rp.lse2 + slot);
      next_tgt = *reinterpret_cast<const LaneInts*>(rp.tgt + slot);
      B.init(p.hidden, p.d, p.gather(), rb * kTile, n_act, p.d, true);
      asm volatile("" : "+v"(next_fac), "+v"(next_lse2), "+v"(next_tgt));
    }
    head_tile<LOADS>(A, p, v0);
    gemm.begin(A, B, smem);
  };
  if (more) begin_tile(chunk * tiles_per_chunk, true);
  while (more) {
    const int n0 = rb * kTile;
    const LaneFloats fac = next_fac, lse2 = next_lse2;
    const LaneInts tgt = next_tgt;
    const int vt_end = min((chunk + 1) * tiles_per_chunk, slab_tiles);
    for (int vt = chunk * tiles_per_chunk; vt < vt_end; ++vt) {
      const int v0 = slab0 + vt * kTile;
      const bool last = vt + 1 == vt_end;
      if (last) units.request();
      GemmAcc<NB> acc;
      gemm.run(A, B, p.d, smem, acc);
      if (last) more = units.next(chunk, rb, &unit_s);
      if (more) begin_tile(last ? chunk * tiles_per_chunk : vt + 1, last);

      bf16* origin = G + (size_t)(v0 - slab0 + uniform(wm)) * p.n_pad + n0 + uniform(wn);
      const unsigned lane_off = (unsigned)(4 * half * p.n_pad + NB * j) * 2u;  // bytes
      // factor * softmax, three instructions per element. (Slots without weight have factor 0 and lse = +inf.)
      const auto store = [&](auto ragged_tile) {
        TileRows rows(origin, p.n_pad * 2);
        int limit = p.V - (v0 + wm + 4 * half);
        if (ragged_tile.value) asm volatile("" : "+v"(limit));
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            LaneFloats x = acc.lane(i, r);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) x[nb] = fac[nb] * exp2_fast(x[nb] * kLog2e - lse2[nb]);
            if (ragged_tile.value && 32 * i + acc_row(r, 0) >= limit) x = LaneFloats{};
            gemm.store(rows, lane_off, r, to_bf16(x));
          }
      };
      if (v0 + kTile > p.V) store(std::true_type{});
      else store(std::false_type{});
      // The targets among the wavefront's elements, of which most column blocks have none, are stored a second time:
      // as a case of every element they cost more than the rest of the epilogue (a tile of 256 x 256 holds one in seven
      // cases of eight at V = 32000; 4096 rows, d = 256: 155 -> 120 us).
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int rel = tgt[nb] - (v0 + wm), row = rel - 4 * half;
        const bool here = (unsigned)rel < (unsigned)kWave && (rel >> 2 & 1) == half;
        if (!__any(here)) continue;
        float logit = 0.f;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float x = acc.value(i, nb, r);
            logit = row == 32 * i + acc_row(r, 0) ? x : logit;
          }
          asm volatile("" : "+v"(logit));
        }
        if (here && fac[nb] != 0.f)
          origin[(size_t)rel * p.n_pad + NB * j + nb] = (bf16)(fac[nb] * (exp2_fast(logit * kLog2e - lse2[nb]) - 1.f));
      }
    }
  }
}

// Same G^T from the f32 logits the forward left in its cache: one pass over memory. A thread
// owns 8 slots and walks kDlogitsRows vocabulary rows with them, so the per-slot constants
// (factor, lse, target: 96 bytes per thread) are loaded once per kDlogitsRows * 32 bytes of
// logits and all of a thread's logits loads are in flight together.
// One thread per (8 vocabulary rows, 8 slots) pair, the slots fastest: at least 32 consecutive lanes
// (n_pad >= 256) read along a row, and no lane idles however few rows there are.
constexpr int kDlogitsRows = 8;
__global__ __launch_bounds__(256) void cutce_dlogits_cached_kernel(CutceParams p, CutceRowParams rp,
                                                                   const float* cache, int slab0,
                                                                   int slab_rows, bf16* G) {
  const int groups = p.n_pad / 8;  // slot groups per vocabulary row
  const long index = (long)blockIdx.x * 256 + threadIdx.x;
  const int vrel0 = (int)(index / groups) * kDlogitsRows;
  const int slot0 = (int)(index % groups) * 8;
  // the two GEMM kernels that follow start from fresh work counters
  if (blockIdx.x == 0) reset_unit_counters(p.header);
  const int n_act = p.header->n_act;
  if (vrel0 >= slab_rows || slot0 >= (n_act + kGemmTile - 1) / kGemmTile * kGemmTile) return;
  const f32x4 f0 = *reinterpret_cast<const f32x4*>(rp.fac + slot0);
  const f32x4 f1 = *reinterpret_cast<const f32x4*>(rp.fac + slot0 + 4);
  const f32x4 l0 = *reinterpret_cast<const f32x4*>(rp.lse2 + slot0);
  const f32x4 l1 = *reinterpret_cast<const f32x4*>(rp.lse2 + slot0 + 4);
  const i32x4 t0 = *reinterpret_cast<const i32x4*>(rp.tgt + slot0);
  const i32x4 t1 = *reinterpret_cast<const i32x4*>(rp.tgt + slot0 + 4);
  f32x4 a[kDlogitsRows], b[kDlogitsRows];
#pragma unroll
  for (int r = 0; r < kDlogitsRows; ++r) {
    // rows past the vocabulary read the last row (the value is not used)
    const float* src = cache + (size_t)min(slab0 + vrel0 + r, p.V - 1) * p.n_pad + slot0;
    a[r] = *reinterpret_cast<const f32x4*>(src);
    b[r] = *reinterpret_cast<const f32x4*>(src + 4);
  }
#pragma unroll
  for (int r = 0; r < kDlogitsRows; ++r) {
    const int v = slab0 + vrel0 + r;
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      out[e] = (bf16)((f0[e] != 0.f && v < p.V) ? dlogit(a[r][e], f0[e], l0[e], t0[e], v) : 0.f);
      out[4 + e] = (bf16)((f1[e] != 0.f && v < p.V) ? dlogit(b[r][e], f1[e], l1[e], t1[e], v) : 0.f);
    }
    store_global16(G + (size_t)(vrel0 + r) * p.n_pad + slot0, as_u32x4(out));
  }
}

// How the two gradient GEMMs of a slab are cut along their contraction. With few rows (or a small
// vocabulary) there are few 256 x 256 output tiles and long contractions: 16 tiles of 32003 terms at
// N = 999, d = 1024, half a millisecond on 16 of 256 compute units. A cut tile leaves f32 partial sums
// [part][rows][columns] that cutce_reduce_kernel adds in part order (deterministic). The number of
// parts is chosen on the device, where the number of active rows is known; the host only
// provides room for them.
struct CutceSplits {
  float* hidden_sums;    // [parts][active row blocks * tile][d]
  float* head_sums;      // [parts][d][slab_width]
  size_t hidden_room;    // floats in hidden_sums
  int head_most;         // parts that head_sums has room for
  int tile;              // 256 or 128: the output tile's sides in this slab
  int head_tile;         // and in a slab of the whole vocabulary
  int vocab;             // columns of the whole vocabulary, padded to 256
  bool with_head;
};

// Lengths in units of 128 terms of one tile: a workgroup's fair share of all of the work is total / slots, and
// tiles much longer than that are cut down to it. Partial sums cost 8 bytes of traffic per part and
// element, so with little work the parts stay longer: at length t the last tile ends after t units and the
// sums take total / t parts, least where t is the square root of total times the price of a part in units
// (256 x 256: 0.1 us of the device's bandwidth against 2 us a unit; 128 x 128: 0.026 against 1).
__host__ __device__ inline float part_length(int tile, int row_blocks, int d, int vocab, bool with_head) {
  const float col_blocks = (float)((d + tile - 1) / tile);
  const float groups = (float)row_blocks * col_blocks * (float)(vocab / 128);
  const float total = (with_head ? 2.f : 1.f) * groups;
  const float share = total / (float)(tile == kGemmTile ? kComputeUnits : 2 * kComputeUnits);
  const float least = __builtin_sqrtf((tile == kGemmTile ? 0.05f : 0.026f) * total);
  return share > least ? share : least;
}
constexpr int kMostParts = 64;
__host__ __device__ inline int whole_parts(float parts) {
  return parts < 1.5f ? 1 : parts > (float)kMostParts ? kMostParts : (int)(parts + 0.5f);
}

CT_DEVICE int hidden_parts(const CutceSplits& sp, int tile, int n_act, int d, int slab_width) {
  const int row_blocks = (n_act + tile - 1) / tile;
  if (row_blocks == 0) return 1;
  const int parts = whole_parts((float)(slab_width / 128) / part_length(tile, row_blocks, d, slab_width, sp.with_head));
  const size_t fit = sp.hidden_room / ((size_t)row_blocks * tile * d);
  return uniform(fit < (size_t)parts ? (fit > 1 ? (int)fit : 1) : parts);
}
// A slab's dHead is cut as the whole vocabulary's is, whatever the slab: dHead is bit for bit the same
// for every workspace. (dHidden adds over slabs anyway.)
CT_DEVICE int head_parts(const CutceSplits& sp, int n_act, int d) {
  const int tile = sp.head_tile;
  const int row_blocks = (n_act + tile - 1) / tile;
  if (row_blocks == 0) return 1;
  const float groups = (float)(row_blocks * (tile / 128));
  return uniform(min(whole_parts(groups / part_length(tile, row_blocks, d, sp.vocab, true)), sp.head_most));
}

// First of the 128-term groups of part `split`.
CT_DEVICE int split_begin(int groups, int split, int splits) { return (int)((long)groups * split / splits); }

// One slab of the vocabulary, as the gradient kernels see it.
struct CutceSlab {
  const bf16* G;       // G^T [width][n_pad]
  const bf16* packed;  // [n_pad][d]
  int first, width;    // vocabulary ids first .. first + width - 1, width a multiple of 256
  int mode;            // 0 = single slab (store bf16), 1 = first slab (store f32), 2 = middle
                       // slab (add f32), 3 = last slab (add, store bf16)
  float* dh_acc;
  bf16* dhidden;
  bf16* dhead;
};

// dHidden[idx[slot], n] (+)= sum_v G^T[v, slot] head[n, first + v] of row block rb, column block cb and
// part `split` of the contraction.
template <int NB, GemmLoads LOADS>
CT_DEVICE void dhidden_unit(const CutceParams& p, const CutceSlab& sl, const CutceSplits& sp, int rb, int cb, int split,
                            int parts, int n_act, UnitQueue& units, const lds_addr smem) {
  constexpr int kTile = GemmShape<NB>::kTile, kWave = GemmShape<NB>::kWave;
  const int tid = threadIdx.x, l = tid & 63, j = l & 31, half = l >> 5, w = tid >> 6;
  const int wm = (w >> 1) * kWave, wn = (w & 1) * kWave;
  // Terms of the contraction: the whole slab where the head is padded, else up to the end of the
  // vocabulary; the last k_width % 128 of them from the tail, since nothing past a row's end may be
  // read (G^T is zero from the vocabulary's end to the end of the slab). The parts are those of the
  // whole slab in each case: the same sums, whether the head is padded or not.
  const int k_width = p.head.padded ? sl.width : min(sl.width, p.V - sl.first), k_whole = k_width / 128 * 128;
  const int groups = sl.width / 128;
  const int n0 = rb * kTile, c0 = cb * kTile;
  const int k_begin = split_begin(groups, split, parts) * 128, k_end = split_begin(groups, split + 1, parts) * 128;
  const int k_mid = min(k_end, k_whole);
  const bool with_tail = k_begin <= k_whole && k_whole < min(k_end, k_width);
  McLoader<NB> A;
  A.init(sl.G, p.n_pad, n0, p.n_pad, sl.width);
  GemmAcc<NB> acc;
  acc.clear();
  // (rows of B interleaved: lane j owns the NB consecutive columns c0 + wn + NB j + nb; rows past d
  // are copies of the first, their columns are not stored)
  const bf16* head = p.head.base + (sl.first - p.head.col0);
  GemmB<NB, LOADS> B;
  if constexpr (LOADS == GemmLoads::kGuarded) {
    B.init(head, p.head.ld, nullptr, c0, p.d, k_width, true);
    gemm_tile<LOADS>(A, B, k_begin, with_tail ? k_width : k_mid, smem, acc);
  } else {
    const bf16* tail = p.head.tail + (sl.first - p.head.tail_first);
#pragma nounroll
    for (int part = 0; part <= (int)with_tail; ++part) {
      B.init(part ? tail : head, part ? p.head.tail_cols : p.head.ld, nullptr, c0, p.d, k_width, true);
      gemm_tile<LOADS>(A, B, part ? k_mid : k_begin, part ? k_mid + 128 : k_mid, smem, acc);
    }
  }
  units.request();

  // To the partial sums or the sum over slabs in f32 (adding what is there from the second slab on), from
  // the only or the last slab to dHidden in bf16. Addresses are a wave-uniform row plus one 32-bit lane
  // offset: formed per element they spill, and a reload waits for every store in front of it (all GEMM
  // epilogues in this form, forward and backward at N = 999, d = 1024, V = 32003: 447 -> 356 us; at N = 16384,
  // d = 4096, V = 128256 part of the 1.6 % that the pass gained in all). Both f32 buffers have rows to the end of the block.
  typedef typename GemmAcc<NB>::Lane LaneFloats;
  typedef decltype(to_bf16(LaneFloats{})) LaneBf16;
  const int row0 = n0 + uniform(wm), col0 = c0 + uniform(wn);
  if (col0 >= p.d) return;  // hidden sizes are multiples of 128: all of the wavefront's columns or none
  if (parts > 1 || sl.mode != 0) {
    float* origin = (parts > 1 ? sp.hidden_sums + (size_t)split * ((n_act + kTile - 1) / kTile * kTile) * p.d
                               : sl.dh_acc) + (size_t)row0 * p.d + col0;
    const unsigned lane_off = (unsigned)(4 * half * p.d + NB * j) * 4u;  // bytes
    TileRows rows(origin, p.d * 4);
    if (parts > 1 || sl.mode == 1) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          store_lane(rows.row, lane_off, acc.lane(i, r));
          rows.advance(r);
        }
      return;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        *reinterpret_cast<LaneFloats*>(rows.row + lane_off) += acc.lane(i, r);
        rows.advance(r);
      }
    if (sl.mode == 2) return;
    for (int r = 0; r < 16 * NB; ++r) {
      const int slot = row0 + 32 * (r >> 4) + acc_row(r & 15, half);
      if (slot >= n_act) continue;
      const LaneFloats val = *reinterpret_cast<const LaneFloats*>(sl.dh_acc + (size_t)slot * p.d + col0 + NB * j);
      *reinterpret_cast<LaneBf16*>(sl.dhidden + (size_t)p.idx[slot] * p.d + col0 + NB * j) = to_bf16(val);
    }
    return;
  }
  bf16* columns = sl.dhidden + col0 + NB * j;
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int slot = row0 + 32 * i + 8 * q + 4 * half;
      const i32x4 to = *reinterpret_cast<const i32x4*>(p.idx + slot);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const LaneBf16 out = to_bf16(acc.lane(i, 4 * q + e));
        if (slot + e < n_act) *reinterpret_cast<LaneBf16*>(columns + (size_t)to[e] * p.d) = out;
      }
    }
}

// Four consecutive columns of a row of dHead; the rows of an odd vocabulary start at any multiple
// of 2 bytes, which an ordinary store may.
CT_DEVICE void store_dhead4(bf16* dst, int left, f32x4 val) {
  bf16x4 out;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) out[nb] = (bf16)val[nb];
  if (left >= 4) {
    __builtin_memcpy(dst, &out, 8);
  } else {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
      if (nb < left) dst[nb] = out[nb];
  }
}

// dHead[m, first + v] = sum_slot packed[slot, m] G^T[v, slot], packed[slot] = hidden[idx[slot]], of
// vocabulary tile vt, hidden column block mb and part `split` of the contraction.
template <int NB, GemmLoads LOADS>
CT_DEVICE void dhead_unit(const CutceParams& p, const CutceSlab& sl, const CutceSplits& sp, int vt, int mb, int split,
                          int parts, int n_act, UnitQueue& units, const lds_addr smem) {
  constexpr int kTile = GemmShape<NB>::kTile, kWave = GemmShape<NB>::kWave;
  const int tid = threadIdx.x, l = tid & 63, j = l & 31, half = l >> 5, w = tid >> 6;
  const int wm = (w >> 1) * kWave, wn = (w & 1) * kWave;
  // 4 contraction steps at a time; slots n_act .. k_end-1 are valid memory: G^T holds zeros
  // there (the dlogits kernels write whole blocks of at least 128 slots) and the packed rows are finite.
  const int groups = min(p.n_pad, (n_act + 4 * kBK - 1) / (4 * kBK) * (4 * kBK)) / (4 * kBK);
  const int m0 = mb * kTile, v0 = vt * kTile;  // v0 relative to the slab
  const int k_begin = split_begin(groups, split, parts) * 128, k_end = split_begin(groups, split + 1, parts) * 128;
  McLoader<NB> A;  // (columns past d are copies, their rows of dHead are not stored)
  A.init(sl.packed, p.d, m0, p.d, k_end);
  // (rows of B interleaved: lane j owns NB consecutive vocabulary ids)
  GemmB<NB, LOADS> B;
  B.init(sl.G, p.n_pad, nullptr, v0, sl.width, k_end, true);
  GemmAcc<NB> acc;
  acc.clear();
  gemm_tile<LOADS>(A, B, k_begin, k_end, smem, acc);
  units.request();

  const int row0 = m0 + uniform(wm), col0 = v0 + uniform(wn);
  if (row0 >= p.d) return;  // hidden sizes are multiples of 128: all of the wavefront's rows or none
  if (parts > 1) {
    float* origin = sp.head_sums + ((size_t)split * p.d + row0) * sl.width + col0;
    const unsigned lane_off = (unsigned)(4 * half * sl.width + NB * j) * 4u;  // bytes
    TileRows rows(origin, sl.width * 4);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        store_lane(rows.row, lane_off, acc.lane(i, r));
        rows.advance(r);
      }
    return;
  }
  // The rows of an odd vocabulary start at any multiple of 2 bytes, which an ordinary store may.
  const int left = p.V - (sl.first + col0 + NB * j);
  bf16* origin = sl.dhead + (size_t)row0 * p.V + sl.first + col0;
  const unsigned lane_off = (unsigned)(4 * half * p.V + NB * j) * 2u;  // bytes
  if (left >= NB) {
    TileRows rows(origin, p.V * 2);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        store_lane(rows.row, lane_off, to_bf16(acc.lane(i, r)));
        rows.advance(r);
      }
  } else {
#pragma unroll
    for (int nb = 0; nb < NB - 1; ++nb)
      if (nb < left) {
        TileRows rows(origin, p.V * 2);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            reinterpret_cast<bf16*>(rows.row + lane_off)[nb] = (bf16)acc.value(i, nb, r);
            rows.advance(r);
          }
      }
  }
}

// Both gradients of a slab in one launch (HEAD = false: the head is frozen). The hidden gradient has few,
// long units (45 x 16 at N = 16384, d = 4096: 2.8 per compute unit, so its last round leaves a sixth of the
// device idle); a workgroup that finds no hidden-gradient unit left goes on to the head-gradient
// units, which are many and short, and the idle tail of the first fills with work of the second. The
// two read the same G^T and write different tensors: neither waits for the other.
template <int NB, bool HEAD, GemmLoads LOADS>
__global__ __launch_bounds__(256, GemmShape<NB>::kGroups) void cutce_grads_kernel(CutceParams p, CutceSlab sl, CutceSplits sp) {
  constexpr int kTile = GemmShape<NB>::kTile;
  extern __shared__ __align__(16) char smem_raw[];
  const lds_addr smem = lds_address_of(smem_raw);
  __shared__ int unit_s;
  const int n_act = p.header->n_act;
  // the dlogits kernel of the next vocabulary slab starts from fresh work counters
  if (blockIdx.x == 0) reset_dlogits_counters(p.header);
  const int col_blocks = (p.d + kTile - 1) / kTile, slab_tiles = sl.width / kTile;
  const int row_blocks = (n_act + kTile - 1) / kTile;
  const int parts_h = hidden_parts(sp, kTile, n_act, p.d, sl.width);
  const int parts_w = HEAD ? head_parts(sp, n_act, p.d) : 1;
  const int total_h = row_blocks * col_blocks * parts_h, total_w = HEAD ? slab_tiles * col_blocks * parts_w : 0;
  // Short problems walk one list, the longer units first; large ones the hidden gradient's grid (row
  // block, (part, column block)) and then the head gradient's (vocabulary tile, (part, column block)).
  const bool one_list = total_h + total_w <= kPlainRounds * (int)gridDim.x;
  // The head's are the longer where there are more rows than vocabulary: few, and last they were alone at the end (both
  // orders, us: 13908 rows x 5376 x 632: 288 / 234, 16384 x 4096 x 1024: 334 / 266, 8000 x 2048 x 2000: 164 / 125; units of
  // about the same length, 5000 x 1024 x 3000: 84 / 87).
  const bool head_first = HEAD && 2l * ((n_act + 127) / 128) * parts_h > 3l * (sl.width / 128) * parts_w;
  UnitQueue units;
  bool in_head = false;
  if (one_list) units.init(p.header->xcd_counter[0], total_h + total_w, 1, UnitQueue::kPlain, true);
  else units.init(p.header->xcd_counter[0], row_blocks, col_blocks * parts_h, UnitQueue::kBlocks);
  for (;;) {
    int a, b;
    if (!units.next(a, b, &unit_s)) {
      if (one_list || in_head || !HEAD) break;
      in_head = true;
      units.init(p.header->xcd_counter[1], slab_tiles, col_blocks * parts_w, UnitQueue::kBlocks);
      continue;
    }
    if (one_list) {
      in_head = head_first ? a < total_w : a >= total_h;
      const int index = a - (in_head == head_first ? 0 : head_first ? total_w : total_h);
      // the part is the slowest: the 32 units of an XCD are all tiles of a few parts, which read the operands' terms of
      // these parts and no others (the tile slowest, an XCD reads all of one operand)
      const int tiles_a = in_head ? slab_tiles : row_blocks, grid = tiles_a * col_blocks;
      const int part = index / grid, tile = index % grid;
      a = tile / col_blocks;
      b = part * col_blocks + tile % col_blocks;
    }
    if (!in_head) {
      dhidden_unit<NB, LOADS>(p, sl, sp, a, b % col_blocks, b / col_blocks, parts_h, n_act, units, smem);
    } else if constexpr (HEAD) {
      // (its operands are the workspace's own)
      constexpr GemmLoads kLoads = LOADS == GemmLoads::kGuarded ? LOADS : GemmLoads::kCopies;
      dhead_unit<NB, kLoads>(p, sl, sp, a, b % col_blocks, b / col_blocks, parts_w, n_act, units, smem);
    }
  }
}

// Adds the partial sums of cut tiles, a thread 4 columns of a row at a time: first those of dHidden's
// active rows, then those of the slab's part of dHead. Nothing to do for a gradient that was not cut.
__global__ __launch_bounds__(256) void cutce_reduce_kernel(CutceParams p, CutceSlab sl, CutceSplits sp) {
  const int n_act = p.header->n_act;
  const long first = (long)blockIdx.x * 256 + threadIdx.x, stride = (long)gridDim.x * 256;
  const int parts_h = hidden_parts(sp, sp.tile, n_act, p.d, sl.width);
  if (parts_h > 1) {
    const int quads = p.d / 4;
    const size_t part_size = (size_t)((n_act + sp.tile - 1) / sp.tile) * sp.tile * p.d;
    for (long index = first; index < (long)n_act * quads; index += stride) {
      const int slot = (int)(index / quads), col = (int)(index % quads) * 4;
      const float* src = sp.hidden_sums + (size_t)slot * p.d + col;
      f32x4 val = *reinterpret_cast<const f32x4*>(src);
#pragma unroll 4
      for (int s = 1; s < parts_h; ++s) val += *reinterpret_cast<const f32x4*>(src + s * part_size);
      f32x4* a = reinterpret_cast<f32x4*>(sl.dh_acc + (size_t)slot * p.d + col);
      if (sl.mode >= 2) val += *a;
      if (sl.mode == 1 || sl.mode == 2) {
        *a = val;
      } else {
        bf16x4 out;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) out[nb] = (bf16)val[nb];
        *reinterpret_cast<bf16x4*>(sl.dhidden + (size_t)p.idx[slot] * p.d + col) = out;
      }
    }
  }
  if (!sp.with_head) return;
  const int parts_w = head_parts(sp, n_act, p.d);
  if (parts_w <= 1) return;
  const int width = min(sl.width, (p.V - sl.first + 3) & ~3);
  const int quads = width / 4;
  for (long index = first; index < (long)p.d * quads; index += stride) {
    const int m = (int)(index / quads), v = (int)(index % quads) * 4;
    const float* src = sp.head_sums + (size_t)m * sl.width + v;
    f32x4 val = *reinterpret_cast<const f32x4*>(src);
#pragma unroll 4
    for (int s = 1; s < parts_w; ++s) val += *reinterpret_cast<const f32x4*>(src + (size_t)s * p.d * sl.width);
    store_dhead4(sl.dhead + (size_t)m * p.V + sl.first + v, p.V - sl.first - v, val);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

static int padded_rows(int N) { return (int)align_up((size_t)N, kGemmTile); }
static int vocab_tile_count(int V) { return (V + kGemmTile - 1) / kGemmTile; }

// Vocabulary tiles per work unit of the two projection kernels. Four keep a unit's hidden rows in use
// for four tiles and leave a quarter of the partial statistics; short problems take units of two
// tiles or one, which end together (263 tiles x 8 row blocks in units of four are 2.06 rounds: three).
static int tiles_per_chunk(int tiles, int row_blocks) {
  const long units = (long)tiles * row_blocks;
  return units <= kPlainRounds * kComputeUnits ? 1 : units <= 2 * kPlainRounds * kComputeUnits ? 2 : 4;
}

// The output tile of the GEMM kernels, 256 or 128. The large one does twice the work per byte that reaches LDS
// (a compute unit's 64 bytes a clock keep up with no more than the small tile's MFMAs); the small one gives
// short problems four times the workgroups, a quarter of the epilogue per wavefront and, up to one tile per
// compute unit, half the time per step. Measured (us, large / small; statistics kernel and dlogits kernel):
// 32 large tiles 500 x 4000, d = 512: 19 / 10 and 20 / 11, d = 6144: 98 / 50 and 100 / 51; 96 large =
// 376 small tiles 1000 x 6000, d = 512: 19 / 17 and 22 / 17, d = 2048: 42 / 40 and 45 / 41; 500 small tiles
// 1000 x 7160, d = 2048: 42 / 41 and 45 / 42, 384 x 19192: 43 / 43 and 46 / 45; 512, 384 x 21880: 47 / 58 and 49 / 60,
// d = 512 21 / 21 and 23 / 24; 704, 4000 x 2800, d = 1024: 30 / 38 and 34 / 40.
constexpr int kMostSmallTiles = 480;
static int projection_tile(int rows, int tiles) {
  return (long)((rows + 127) / 128) * (2 * tiles) <= kMostSmallTiles ? 128 : kGemmTile;
}
// The gradients cut long contractions, so the large tile fills the device too, at the price of more partial sums.
// By the groups of 128 terms of all small tiles (with the reduction; large / small): 384 of them 300 x 776, d = 1024:
// 23 / 15; 1024, 500 x 4000, d = 512: 25 / 20; 2048, 500 x 8000: 28 / 26; 3072, 1000 x 6000: 31 / 33; 4096,
// 500 x 4000, d = 2048: 36 / 40.
constexpr int kMostSmallGroups = 1536;
static int gradient_tile(const ct_cutce_shape& s) {
  const long groups = 2L * ((s.rows + 127) / 128) * (s.hidden / 128) * (2 * vocab_tile_count(s.vocab));
  return groups <= kMostSmallGroups ? 128 : kGemmTile;
}

// The statistics kernel's units: `chunks` of `per_chunk` tiles of `tile` columns.
struct StatsUnits {
  int tile, tiles, per_chunk, chunks;
};
static StatsUnits stats_units(const ct_cutce_shape& s) {
  const int tiles = vocab_tile_count(s.vocab), row_blocks = padded_rows(s.rows) / kGemmTile;
  if (projection_tile(s.rows, tiles) != kGemmTile) {
    const int small = (s.vocab + 127) / 128;
    return {128, small, 1, small};
  }
  const int t = tiles_per_chunk(tiles, row_blocks);
  return {kGemmTile, tiles, t, (tiles + t - 1) / t};
}

// Heads whose rows do not all start on 16 bytes go through an aligned copy (HeadCopy).
static bool needs_panel(const ct_cutce_shape& s) { return s.vocab % 8 != 0; }
// ... or are read in place by loads through registers, which need a copy of the last columns only (HeadView::tail). The copy
// of the whole takes 4 bytes of traffic per element and direction, and leaves aligned 16-byte chunks: unaligned ones make
// a product 5 to 15 % longer (24 % where two small tiles share a compute unit), so it pays from some number of
// rows on. Us, copy / in place, one GPU.
// Forward (copy and statistics kernel): 128 x 150001, d = 4096 768 / 340; 250 x 50001, d = 1024 74 / 38; 1000 x 16001,
// d = 1024 46 / 42; 2000 x 50001, d = 4096 833 / 811, d = 256 98 / 97; 4000 x 50001, d = 1024 417 / 428, d = 256 165 / 175. Fewer
// than 8 columns per row: 1000 x 5001, d = 4096 79 / 85, d = 1024 28.0 / 30.5; a chain along d longer than the copy: 128 x
// 1501, d = 4096 41 / 44, d = 1024 19.0 / 16.5.
static bool forward_in_place(const ct_cutce_shape& s) {
  return needs_panel(s) && s.rows <= 2048 && s.vocab >= 8l * s.rows && 2l * s.vocab >= s.hidden;
}
// Backward (copy, dlogits and gradients), where dHidden reads short rows: 64 x 150001, d = 4096 1466 / 1165, d = 256 163 / 132;
// 250 x 50001, d = 1024 149 / 122; 512 x 100003, d = 1024 418 / 391, x 50257, d = 4096 747 / 696. The larger the head, the fewer the
// rows that it pays for: 640 x 50257, d = 2048 491 / 510, x 16001, d = 8192 646 / 720; 768 x 50257, d = 1024 273 / 264, x 16001, d = 4096
// 316 / 301, x 100003, d = 512 296 / 303; 1024 x 150001, d = 256 340 / 353, x 50257, d = 1024 333 / 348, x 32003, d = 2048 382 / 393, but
// x 16001, d = 2048 213 / 194, x 32003, d = 512 129 / 126; 1280 x 16001, d = 1024 147 / 155, d = 2048 268 / 264; 2048 x 16001, d = 1024
// 190 / 202, x 150001, d = 256 605 / 656. Small heads: 64 x 16001, d = 256 31.2 / 32.0, 500 x 5001, d = 1024 46.8 / 50.6.
static bool backward_in_place(const ct_cutce_shape& s) {
  const long elements = (long)s.hidden * s.vocab;
  const int most_rows = elements <= 35000000 ? 1024 : elements <= 100000000 ? 768 : 512;
  return needs_panel(s) && s.vocab >= 8192 && elements >= 12000000 && s.rows <= most_rows;
}
// With a logits cache or a kept panel one copy serves both directions, so it has to be paid for once only, and reading in place is
// ahead of it for fewer calls. A pass with both buffers allowed, copy / in place: 64 x 32003, d = 4096 360 / 287; 512 x 16001, d = 1024
// 117 / 115, x 100003 535 / 491, d = 512 331 / 312, x 150001 448 / 441; up to 35 million elements at 1024 rows too: x 50257, d = 256
// 206 / 196, x 32003, d = 512 183 / 183, x 16001, d = 2048 252 / 234; not beyond: 1024 x 100003, d = 512 508 / 525, x 150001 712 / 756,
// 640 x 100003, d = 768 521 / 551, x 32003, d = 2048 374 / 397.
static bool both_in_place(const ct_cutce_shape& s) {
  return forward_in_place(s) && backward_in_place(s) && (s.rows <= 512 || (long)s.hidden * s.vocab <= 35000000);
}
static size_t panel_tile_bytes(const ct_cutce_shape& s) { return (size_t)s.hidden * kGemmTile * sizeof(bf16); }
// bytes of the panel of the whole vocabulary, 0 if none is needed
static size_t full_panel_bytes(const ct_cutce_shape& s) {
  return needs_panel(s) ? panel_tile_bytes(s) * vocab_tile_count(s.vocab) : 0;
}
// What a direction makes of an unaligned head: read in place, the tail only.
static size_t copy_bytes(const ct_cutce_shape& s, bool in_place) { return in_place ? panel_tile_bytes(s) : full_panel_bytes(s); }

// Workspace of the forward: `base` bytes it cannot do without, then as much of the panel as fits, or the tail.
struct FwdLayout {
  size_t header, idx, target, active, part, sums, base, total;
};
static FwdLayout fwd_layout(const ct_cutce_shape& s) {
  const int n_pad = padded_rows(s.rows);
  FwdLayout L;
  L.header = 0;
  L.idx = align_up(sizeof(CutceHeader), 256);
  L.target = L.idx + align_up((size_t)n_pad * sizeof(int), 256);
  L.active = L.target + align_up((size_t)n_pad * sizeof(int), 256);
  L.part = L.active + align_up((size_t)(n_pad / kGemmTile) * sizeof(int), 256);
  L.sums = L.part + align_up((size_t)stats_units(s).chunks * n_pad * 3 * sizeof(float), 256);
  L.base = L.sums + align_up((size_t)(n_pad / kMergeSlots) * 2 * sizeof(double), 256);
  L.total = L.base + full_panel_bytes(s);
  return L;
}

// Room for the partial sums (see CutceSplits). The bytes that the parts of dHidden take, and the number
// of parts of dHead, are largest with every row active (times 4/3: a number of parts is rounded).
// Short problems get the room of both tiles: the large one cuts them into more parts, and a caller's bound on
// the workspace that is a share of the preferred size (local_chunk_size) stays what it was.
static size_t hidden_sums_bytes(const ct_cutce_shape& s, int tile, int slab_tiles, bool with_head) {
  const int row_blocks = (s.rows + tile - 1) / tile, width = slab_tiles * kGemmTile;
  const double parts = (double)(width / 128) / part_length(tile, row_blocks, s.hidden, width, with_head);
  const double least = 1.5 / row_blocks;  // with fewer not even a single row block is cut
  return parts < least ? 0 : align_up((size_t)(1.34 * parts * row_blocks * tile * s.hidden * sizeof(float)), 256);
}
static size_t hidden_sums_bytes(const ct_cutce_shape& s, int slab_tiles, bool with_head) {
  const size_t large = hidden_sums_bytes(s, kGemmTile, slab_tiles, with_head);
  const size_t chosen = hidden_sums_bytes(s, gradient_tile(s), slab_tiles, with_head);
  return large > chosen ? large : chosen;
}
// What kMostParts parts take, with the tile of a slab of this size: more room than that is never used.
static size_t most_hidden_sums_bytes(const ct_cutce_shape& s, int slab_tiles) {
  const int tile = gradient_tile(ct_cutce_shape{s.rows, s.hidden, slab_tiles * kGemmTile});
  return (size_t)kMostParts * ((s.rows + tile - 1) / tile) * tile * s.hidden * sizeof(float);
}
static int most_head_parts(const ct_cutce_shape& s, int tile) {
  const int row_blocks = (s.rows + tile - 1) / tile;
  return whole_parts((float)(row_blocks * (tile / 128)) /
                     part_length(tile, row_blocks, s.hidden, vocab_tile_count(s.vocab) * kGemmTile, true));
}
static int most_head_parts(const ct_cutce_shape& s) {
  return max(most_head_parts(s, kGemmTile), most_head_parts(s, gradient_tile(s)));
}

struct BwdLayout {
  size_t header, idx, rowparams, packed, tail, panel, g, head_sums, acc, hidden_sums, total;
  size_t hidden_sums_bytes;
  int head_most;
  int slab_cols;  // multiple of 256
  int slabs;
};
// header, idx, 3 row parameter arrays, packed hidden rows, tail of the head
static size_t bwd_fixed_bytes(int n_pad, int d) {
  return align_up(sizeof(CutceHeader), 256) + 4 * align_up((size_t)n_pad * sizeof(int), 256) +
         align_up((size_t)n_pad * d * sizeof(bf16), 256) + (size_t)d * 128 * sizeof(bf16);
}
// What one tile column of a slab takes: its part of G^T, its columns of a head that is copied here, and the partial
// sums of dHead if that is cut.
struct BwdTileBytes {
  size_t g, panel, head_sums;
  size_t all() const { return g + panel + head_sums; }
};
// What the workspace of the backward holds of an unaligned head: copies of the slabs' columns, the tail, or nothing (the panel is lent
// or in the logits cache). With the tail the copies' bytes go to wider slabs and more parts. A bounded call that copies slab by
// slab / reads in place, us of a pass: 144 x 30159, d = 2432 in chunks of 24 rows 494 / 237, 64 x 50257, d = 1024 by 4 568 / 269,
// 512 x 32003, d = 4096 by 85 955 / 575, 999 x 32003, d = 1024 by 166 506 / 441, 900 x 50257, d = 256 by 450 211 / 219.
enum class HeadPart { kPanel, kTail, kNothing };
static HeadPart bwd_head_part(const ct_cutce_shape& s, bool panel_elsewhere) {
  return !needs_panel(s) || panel_elsewhere ? HeadPart::kNothing : backward_in_place(s) ? HeadPart::kTail : HeadPart::kPanel;
}
static BwdTileBytes bwd_tile_bytes(const ct_cutce_shape& s, HeadPart part, bool with_head) {
  const int parts = with_head ? most_head_parts(s) : 1;
  return BwdTileBytes{(size_t)padded_rows(s.rows) * kGemmTile * sizeof(bf16), part == HeadPart::kPanel ? panel_tile_bytes(s) : 0,
                      parts > 1 ? (size_t)parts * s.hidden * kGemmTile * sizeof(float) : 0};
}
static size_t bwd_acc_bytes(const ct_cutce_shape& s) {
  return align_up((size_t)padded_rows(s.rows) * s.hidden * sizeof(float), 256);
}
// Estimated time (us) of a backward in slabs of `slab_tiles` tile columns with `spare` bytes for the partial sums of dHidden. A
// group of 128 terms of a tile takes 2 us (256 x 256; 1.5 where a hidden size of 128 leaves half of it empty) or 1 (128 x 128). A
// dHidden unit walks all groups of its part, of which there are kMostParts at most: without room for parts a slab's few units
// leave the device idle (704 rows x 1152 x 41694 in four slabs: ten units of 160 us). A dHead unit walks its part of the
// rows in every slab, however narrow, in parts that the whole vocabulary has set; those chains have the device almost to themselves and
// take 0.6 of the time per group. A slab pays for four launches, for large sums to write, read and add (8 bytes per part and element, at
// 5 TB/s) and, in its dlogits, for one walk along the hidden size at least. Us of a pass with the chains, the large sums and the
// most parts left out / counted, and the largest slab that fits: 4180 x 896 x 42590 in chunks of 469 rows 1950 / 1390, 1390;
// 4270 x 512 x 26982 by 439 1595 / 895, 898; 9149 x 256 x 8364 by 1887 513 / 400, 509; 3556 x 256 x 89215 by 297 1464 / 1247, 1818;
// 13 x 256 x 102429 by 10, frozen head, 114 / 97, 97; 100 drawn shapes where the choice differs 0.56 to 1.12 times, 0.92 in the mean.
static float slabs_time(const ct_cutce_shape& s, int slab_tiles, size_t spare, bool with_head) {
  const int tile = gradient_tile(ct_cutce_shape{s.rows, s.hidden, slab_tiles * kGemmTile}), head_tile = gradient_tile(s);
  const int row_blocks = (s.rows + tile - 1) / tile, col_blocks = (s.hidden + tile - 1) / tile;
  const float group = tile != kGemmTile ? 1.f : s.hidden > 128 ? 2.f : 1.5f;
  const float slots = (float)(tile == kGemmTile ? kComputeUnits : 2 * kComputeUnits), groups = 2.f * slab_tiles;
  const float want = groups / part_length(tile, row_blocks, s.hidden, slab_tiles * kGemmTile, with_head);
  const float fit = (float)(spare / ((size_t)row_blocks * tile * s.hidden * sizeof(float)));
  const float parts = fmaxf(1.f, fminf(fminf(want, (float)kMostParts), fit));
  const float row_groups = (float)((s.rows + head_tile - 1) / head_tile * (head_tile / 128));
  const float head_chain = with_head ? 0.6f * row_groups / most_head_parts(s, head_tile) : 0.f;
  const float all = (with_head ? 2.f : 1.f) * row_blocks * col_blocks * groups / slots;
  const float sums = (parts < 1.5f ? 1.f : 1.f + parts) * s.rows * s.hidden * (8.f / 5e6f);
  const float slab = fmaxf(fmaxf(groups / parts, head_chain), all) * group + fmaxf(20.f, 5.f + sums) + s.hidden / 128.f;
  return slab * ((vocab_tile_count(s.vocab) + slab_tiles - 1) / slab_tiles);
}
// The whole vocabulary as one slab if that fits in `bytes` with room for all parts of dHidden behind it, else the size
// of a slab that takes the least time (slab_cols = 0 if not even one tile column fits). The partial sums of a cut
// dHidden come last: as many parts as fit behind a slab. The largest slab that fits, or one down to half
// of it where all parts then fit, and the present size (us of a pass): 638 x 256 x 133066 in chunks of 36 rows, 18 slabs now, 2500 / 709,
// 84 x 2432 x 132192 by 22, 4, 3516 / 913, 290 x 768 x 141343 by 32, frozen head, 12, 2420 / 732, 456 x 256 x 24749 by 23, 14,
// 432 / 388, 5058 x 1024 x 108442 by 125, 39, 5105 / 5100.
static BwdLayout bwd_layout(const ct_cutce_shape& s, size_t bytes, bool panel_elsewhere, bool with_head) {
  const HeadPart part = bwd_head_part(s, panel_elsewhere);
  const int n_pad = padded_rows(s.rows);
  const int tiles = vocab_tile_count(s.vocab);
  BwdLayout L = {};
  L.header = 0;
  L.idx = align_up(sizeof(CutceHeader), 256);
  L.rowparams = L.idx + align_up((size_t)n_pad * sizeof(int), 256);
  L.packed = L.rowparams + 3 * align_up((size_t)n_pad * sizeof(int), 256);
  L.panel = bwd_fixed_bytes(n_pad, s.hidden);
  L.tail = L.panel - (size_t)s.hidden * 128 * sizeof(bf16);
  const BwdTileBytes tile = bwd_tile_bytes(s, part, with_head);
  const size_t per_tile = tile.all(), acc_bytes = bwd_acc_bytes(s);
  const size_t slab = L.panel + (part == HeadPart::kTail ? panel_tile_bytes(s) : 0);  // where a slab's part begins
  size_t fit = tiles, room;
  L.head_most = with_head ? most_head_parts(s) : 1;
  const bool whole = bytes >= slab + per_tile * tiles;
  room = whole ? bytes - slab : 0;
  const size_t all_sums = std::min(hidden_sums_bytes(s, tiles, with_head), most_hidden_sums_bytes(s, tiles));
  if (!whole || room - per_tile * tiles < all_sums) {
    float least = whole ? slabs_time(s, tiles, room - per_tile * tiles, with_head) : __builtin_inff();
    const size_t slabs_room = bytes < slab + acc_bytes ? 0 : bytes - slab - acc_bytes;
    const size_t most = slabs_room / per_tile;
    if (!whole && most == 0) return L;
    for (size_t fewer = most < (size_t)tiles ? most : (size_t)tiles - 1; fewer > 0; fewer -= (fewer + 7) / 8) {
      const float time = slabs_time(s, (int)fewer, slabs_room - per_tile * fewer, with_head);
      if (time >= least) continue;
      least = time;
      fit = fewer;
      room = slabs_room;
    }
  }
  const size_t want = hidden_sums_bytes(s, (int)fit, with_head), spare = (room - per_tile * fit) / 256 * 256;
  L.hidden_sums_bytes = want < spare ? want : spare;
  L.slab_cols = (int)fit * kGemmTile;
  L.slabs = (tiles + (int)fit - 1) / (int)fit;
  L.g = slab + tile.panel * fit;
  L.head_sums = L.g + tile.g * fit;
  L.acc = L.head_sums + tile.head_sums * fit;
  L.hidden_sums = L.acc + (L.slabs > 1 ? acc_bytes : 0);
  L.total = L.hidden_sums + L.hidden_sums_bytes;
  return L;
}

static int validate_cutce(const char* fn, const ct_cutce_shape& s) {
  CT_REQUIRE(s.rows > 0, "%s: Cut cross-entropy requires at least one token row", fn);
  CT_REQUIRE(s.hidden > 0 && s.hidden % 128 == 0,
             "%s: Cut cross-entropy hidden size must be divisible by 128, got %d", fn, s.hidden);
  CT_REQUIRE(s.vocab > 0, "%s: Cut cross-entropy requires a non-empty vocabulary", fn);
  return CT_OK;
}

// The GEMM loop addresses the 256 rows of a k-contiguous tile by 32-bit byte offsets (KcLoader::voff).
// Rows in place are offsets from the tile's first row, so it is their stride that is limited ...
constexpr int kMaxRowStride = 1 << 23;  // elements: 255 rows of 2 bytes each stay below 4 GiB
// ... and gathered rows are offsets from the tensor's first.
static bool gather_reaches(const ct_cutce_shape& s) {
  return (size_t)s.rows * (size_t)s.hidden * sizeof(bf16) <= (size_t)1 << 32;
}
// The gradients read such tiles of the head (stride: its padded vocabulary) and, for dHead, of G^T
// (stride: its padded rows).
static int validate_cutce_strides(const char* fn, const ct_cutce_shape& s, bool with_head) {
  if (vocab_tile_count(s.vocab) > kMaxRowStride / kGemmTile || (with_head && s.rows > kMaxRowStride))
    return fail(CT_UNSUPPORTED, "%s: a vocabulary of more than 2^23 (got %d), or dHead over more than 2^23 rows (got %d)",
                fn, s.vocab, s.rows);
  return CT_OK;
}

static bool is_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The GEMM kernels need more than the default 64 KB of LDS; each says so once per device.
template <class... Kernels>
static int allow_gemm_lds(const char* fn, std::atomic<unsigned>& done, Kernels... kernels) {
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 32) device = -1;
  if (device >= 0 && (done.load(std::memory_order_acquire) >> device & 1u)) return CT_OK;
  for (const void* kernel : {reinterpret_cast<const void*>(kernels)...}) {
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)GemmShape<4>::kBytes);
    if (e != hipSuccess) return fail(CT_LAUNCH_FAILED, "%s: %s", fn, hipGetErrorString(e));
  }
  if (device >= 0) done.fetch_or(1u << device, std::memory_order_release);
  return CT_OK;
}

// Compute units of the current device, asked for once per device.
static int device_cu_count() {
  static std::atomic<int> known[32];
  int device = 0, cus = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 32) return kComputeUnits;
  if ((cus = known[device].load(std::memory_order_relaxed)) > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = kComputeUnits;
  known[device].store(cus, std::memory_order_relaxed);
  return cus;
}

}  // namespace ct

using namespace ct;

static bool valid_sizes(const ct_cutce_shape* s) { return s && s->rows > 0 && s->hidden > 0 && s->vocab > 0; }

extern "C" size_t ct_cutce_fwd_workspace_bytes(const ct_cutce_shape* shape) {
  return valid_sizes(shape) ? fwd_layout(*shape).total : 0;
}

extern "C" size_t ct_cutce_fwd_workspace_used_bytes(const ct_cutce_shape* shape) {
  return valid_sizes(shape) ? fwd_layout(*shape).base + copy_bytes(*shape, forward_in_place(*shape)) : 0;
}

extern "C" size_t ct_cutce_fwd_workspace_min_bytes(const ct_cutce_shape* shape) {
  return valid_sizes(shape) ? fwd_layout(*shape).base : 0;
}

namespace ct {
static size_t logits_bytes(const ct_cutce_shape& s) {
  return (size_t)padded_rows(s.rows) * vocab_tile_count(s.vocab) * kGemmTile * sizeof(float);
}
}  // namespace ct

extern "C" size_t ct_cutce_logits_cache_bytes(const ct_cutce_shape* shape) {
  return valid_sizes(shape) ? logits_bytes(*shape) + full_panel_bytes(*shape) : 0;
}

extern "C" size_t ct_cutce_logits_cache_used_bytes(const ct_cutce_shape* shape) {
  return valid_sizes(shape) ? logits_bytes(*shape) + copy_bytes(*shape, both_in_place(*shape)) : 0;
}

extern "C" size_t ct_cutce_bwd_workspace_used_bytes(const ct_cutce_shape* shape) {
  if (!valid_sizes(shape)) return 0;
  const size_t trained = bwd_layout(*shape, ~(size_t)0, false, true).total;
  const size_t frozen = bwd_layout(*shape, ~(size_t)0, false, false).total;
  return trained > frozen ? trained : frozen;
}

extern "C" size_t ct_cutce_bwd_workspace_bytes(const ct_cutce_shape* shape) {
  if (!valid_sizes(shape)) return 0;
  return ct_cutce_bwd_workspace_used_bytes(shape) + full_panel_bytes(*shape) - copy_bytes(*shape, backward_in_place(*shape));
}

extern "C" size_t ct_cutce_bwd_workspace_min_bytes(const ct_cutce_shape* shape) {
  if (!valid_sizes(shape)) return 0;
  const size_t fixed =
      bwd_fixed_bytes(padded_rows(shape->rows), shape->hidden) + bwd_tile_bytes(*shape, HeadPart::kNothing, true).all() +
      (needs_panel(*shape) ? panel_tile_bytes(*shape) : 0);  // (one column of the panel, or the tail)
  return vocab_tile_count(shape->vocab) == 1 ? fixed : fixed + bwd_acc_bytes(*shape);
}

static CutceParams make_params(const uint16_t* hidden, const uint16_t* head, const int32_t* targets,
                               const float* weights, const ct_cutce_shape& s, int compact, char* ws) {
  CutceParams p = {};
  p.hidden = reinterpret_cast<const bf16*>(hidden);
  p.head = HeadView{reinterpret_cast<const bf16*>(head), nullptr, s.vocab, 0, 0, 0, false};
  p.compact = compact && gather_reaches(s);  // (rows in place give the same results)
  p.targets = targets;
  p.weights = weights;
  p.N = s.rows;
  p.d = s.hidden;
  p.V = s.vocab;
  p.n_pad = padded_rows(s.rows);
  p.header = reinterpret_cast<CutceHeader*>(ws);
  p.idx = reinterpret_cast<int*>(ws + align_up(sizeof(CutceHeader), 256));
  p.hidden_aligned = is_aligned16(hidden);
  return p;
}

// The row list in `list_blocks` workgroups and a copy of the head (either may be nothing).
template <bool BACKWARD>
static int launch_prepare(hipStream_t stream, const CutceParams& p, const CutceRowWork& work, const HeadCopy& copy,
                          int list_blocks, bool reset) {
  LaunchScope scope("cutce_prepare_kernel", stream);
  hipLaunchKernelGGL(cutce_prepare_kernel<BACKWARD>, dim3(list_blocks + head_copy_blocks(copy, p.d)), dim3(1024), 0, stream, p,
                     work, copy, list_blocks, reset);
  return scope.done();
}
// `panel` with the tile columns tile0 .. tile0 + tiles - 1 of the head.
static HeadCopy panel_copy(const bf16* head, bf16* panel, int tile0, int tiles) {
  return HeadCopy{head, panel, nullptr, tile0 * kGemmTile, tiles * kGemmTile, 0, 0};
}
static HeadView panel_view(const bf16* panel, int tile0, int tiles) {
  return HeadView{panel, nullptr, (long)tiles * kGemmTile, tile0 * kGemmTile, 0, 0, true};
}
// A view of the caller's head with a tail of `cols` columns, and the copy that fills it.
static HeadView tail_view(const CutceParams& p, const bf16* tail, int cols) {
  return HeadView{p.head.base, tail, p.V, 0, p.V / cols * cols, cols, false};
}
static HeadCopy tail_copy(const HeadView& view) {
  return HeadCopy{view.base, nullptr, const_cast<bf16*>(view.tail), 0, 0, view.tail_first, view.tail_cols};
}

constexpr GemmLoads kCopies = GemmLoads::kCopies, kThrough = GemmLoads::kThroughRegisters, kGuarded = GemmLoads::kGuarded;
template <class Kernel>
static Kernel by_loads(GemmLoads loads, Kernel copies, Kernel through, Kernel guarded) {
  return loads == kCopies ? copies : loads == kThrough ? through : guarded;
}

// Launches of no more small tiles than compute units: a workgroup has its compute unit to itself, its copies are its own
// latency, and with twice the LDS they are on their way for six steps instead of two. Statistics kernel, four / eight stages,
// us: 588 x 1248, d = 6400 (50 tiles) 48.5 / 42.0; 1393 x 704, d = 5504 (66) 43.9 / 36.8; 385 x 3120, d = 7296 (100)
// 56.3 / 49.3; 69 x 5667, d = 1536 (45) 20.4 / 17.4; a contraction that is over in a few steps pays for the longer
// start: 64 x 600, d = 256 7.9 / 8.6.
static bool alone(int units, int hidden, GemmLoads loads) { return units <= device_cu_count() && hidden >= 768 && loads != kGuarded; }

template <int NB, int RING = 4>
static int launch_stats(const char* fn, hipStream_t stream, const CutceParams& p, GemmLoads loads, float* part, int chunk0,
                        int chunks, int tiles_per_chunk, float* cache) {
  const int units = chunks * ((p.N + 64 * NB - 1) / (64 * NB));
  if constexpr (NB == 2 && RING == 4)
    if (alone(units, p.d, loads)) return launch_stats<2, 8>(fn, stream, p, loads, part, chunk0, chunks, tiles_per_chunk, cache);
  constexpr GemmLoads kAny = RING == 4 ? kGuarded : kCopies;
  static std::atomic<unsigned> lds_allowed{0};
  const int rc = allow_gemm_lds(fn, lds_allowed, cutce_stats_kernel<NB, false, kCopies, RING>, cutce_stats_kernel<NB, true, kCopies, RING>,
                                cutce_stats_kernel<NB, false, kThrough, RING>, cutce_stats_kernel<NB, true, kThrough, RING>,
                                cutce_stats_kernel<NB, false, kAny, RING>, cutce_stats_kernel<NB, true, kAny, RING>);
  if (rc) return rc;
  const auto kernel = cache ? by_loads(loads, cutce_stats_kernel<NB, true, kCopies, RING>, cutce_stats_kernel<NB, true, kThrough, RING>,
                                       cutce_stats_kernel<NB, true, kAny, RING>)
                            : by_loads(loads, cutce_stats_kernel<NB, false, kCopies, RING>, cutce_stats_kernel<NB, false, kThrough, RING>,
                                       cutce_stats_kernel<NB, false, kAny, RING>);
  typedef GemmShape<NB, RING> Shape;
  LaunchScope scope("cutce_stats_kernel", stream);
  hipLaunchKernelGGL(kernel, dim3(min(device_cu_count() * Shape::kGroups, units)), dim3(256), Shape::kBytes, stream, p, part, chunk0,
                     chunks, tiles_per_chunk, cache);
  return scope.done();
}

// slab_tiles: of the kernel's tile size
template <int NB, int RING = 4>
static int launch_dlogits(const char* fn, hipStream_t stream, const CutceParams& p, const CutceRowParams& rp, GemmLoads loads,
                          int slab0, int slab_tiles, int tiles_per_chunk, bf16* G) {
  const int units = (slab_tiles + tiles_per_chunk - 1) / tiles_per_chunk * ((p.N + 64 * NB - 1) / (64 * NB));
  if constexpr (NB == 2 && RING == 4)
    if (alone(units, p.d, loads)) return launch_dlogits<2, 8>(fn, stream, p, rp, loads, slab0, slab_tiles, tiles_per_chunk, G);
  constexpr GemmLoads kAny = RING == 4 ? kGuarded : kCopies;
  static std::atomic<unsigned> lds_allowed{0};
  const int rc = allow_gemm_lds(fn, lds_allowed, cutce_dlogits_kernel<NB, kCopies, RING>, cutce_dlogits_kernel<NB, kThrough, RING>,
                                cutce_dlogits_kernel<NB, kAny, RING>);
  if (rc) return rc;
  typedef GemmShape<NB, RING> Shape;
  LaunchScope scope("cutce_dlogits_kernel", stream);
  hipLaunchKernelGGL(by_loads(loads, cutce_dlogits_kernel<NB, kCopies, RING>, cutce_dlogits_kernel<NB, kThrough, RING>,
                              cutce_dlogits_kernel<NB, kAny, RING>),
                     dim3(min(device_cu_count() * Shape::kGroups, units)), dim3(256), Shape::kBytes, stream, p, rp, slab0, slab_tiles,
                     tiles_per_chunk, G);
  return scope.done();
}

template <int NB>
static int launch_grads(const char* fn, hipStream_t stream, const CutceParams& p, const CutceSlab& slab, const CutceSplits& sp,
                        GemmLoads loads) {
  static std::atomic<unsigned> lds_allowed{0};
  const int rc = allow_gemm_lds(fn, lds_allowed, cutce_grads_kernel<NB, false, kCopies>, cutce_grads_kernel<NB, true, kCopies>,
                                cutce_grads_kernel<NB, false, kThrough>, cutce_grads_kernel<NB, true, kThrough>,
                                cutce_grads_kernel<NB, false, kGuarded>, cutce_grads_kernel<NB, true, kGuarded>);
  if (rc) return rc;
  const auto kernel = sp.with_head ? by_loads(loads, cutce_grads_kernel<NB, true, kCopies>, cutce_grads_kernel<NB, true, kThrough>,
                                              cutce_grads_kernel<NB, true, kGuarded>)
                                   : by_loads(loads, cutce_grads_kernel<NB, false, kCopies>, cutce_grads_kernel<NB, false, kThrough>,
                                              cutce_grads_kernel<NB, false, kGuarded>);
  LaunchScope scope(sp.with_head ? "cutce_grads_kernel" : "cutce_dhidden_kernel", stream);
  hipLaunchKernelGGL(kernel, dim3(device_cu_count() * GemmShape<NB>::kGroups), dim3(256), GemmShape<NB>::kBytes, stream, p, slab,
                     sp);
  return scope.done();
}

// The panel and the logits cache that a caller lends. A cache has room for a panel (or a tail) behind its logits, which a
// forward with a lent panel would leave unwritten, so with one the cache ends behind the logits: the entries
// without a panel refuse it as too small.
static int validate_lent(const char* fn, const ct_cutce_shape& s, const void* panel, size_t panel_bytes, const void* cache,
                         size_t cache_bytes) {
  const bool lent = panel && needs_panel(s);
  CT_REQUIRE(!lent || is_aligned16(panel), "%s: panel must be 16-byte aligned", fn);
  if (lent && panel_bytes < full_panel_bytes(s))
    return fail(CT_WORKSPACE_TOO_SMALL, "%s: panel %zu < %zu bytes", fn, panel_bytes, full_panel_bytes(s));
  if (!cache) return CT_OK;
  CT_REQUIRE(is_aligned16(cache), "%s: logits cache must be 16-byte aligned", fn);
  const size_t need = logits_bytes(s) + (lent ? 0 : copy_bytes(s, both_in_place(s)));
  if (cache_bytes < need) return fail(CT_WORKSPACE_TOO_SMALL, "%s: logits cache %zu < %zu bytes", fn, cache_bytes, need);
  CT_REQUIRE(!lent || cache_bytes == need, "%s: beside a panel the logits cache is %zu bytes, without room for one, not %zu", fn,
             need, cache_bytes);
  return CT_OK;
}

// Shared body of ct_cutce_fwd and ct_cutce_fwd_noalloc: `ws` / `ws_bytes` is the workspace to use
// (the caller's, or this device's static scratch array), `fn` the name for error texts.
// `lent`: the caller's panel or null, made here unless `filled`.
static int32_t cutce_fwd_on(void* stream_, const ct_cutce_fwd_args* a, void* ws_, size_t ws_bytes,
                            const char* fn, bf16* lent = nullptr, size_t lent_bytes = 0, bool filled = false) {
  CT_REQUIRE(a->hidden && a->head && a->targets && a->weights && a->nll_sum && a->weight_sum &&
                 a->lse && ws_,
             "%s: null pointer", fn);
  int rc = validate_cutce(fn, a->shape);
  if (rc) return rc;
  const FwdLayout L = fwd_layout(a->shape);
  if (ws_bytes < L.base)
    return fail(CT_WORKSPACE_TOO_SMALL, "%s: workspace %zu < %zu bytes", fn, ws_bytes, L.base);
  CT_REQUIRE(is_aligned16(ws_), "%s: workspace must be 16-byte aligned", fn);
  if ((rc = validate_lent(fn, a->shape, lent, lent_bytes, a->logits_cache, a->logits_cache_bytes))) return rc;
  hipStream_t stream = (hipStream_t)stream_;
  char* ws = static_cast<char*>(ws_);
  CutceParams p = make_params(a->hidden, a->head, a->targets, a->weights, a->shape, a->sparse_compaction, ws);
  float* part = reinterpret_cast<float*>(ws + L.part);
  double* sums = reinterpret_cast<double*>(ws + L.sums);
  const bf16* head = p.head.base;

  p.slot_target = reinterpret_cast<int*>(ws + L.target);
  p.block_active = reinterpret_cast<int*>(ws + L.active);
  const StatsUnits units = stats_units(a->shape);
  // The panel of a head with unaligned rows: lent by the caller, at the end of the logits cache, where the backward finds
  // it again, or in what the workspace has behind its fixed part, a number of chunks at a time.
  const int step_tiles = units.per_chunk, step_chunks = kGemmTile / units.tile;  // 256-column tiles and chunks of a panel step
  // Read in place it needs the panel's first tile column only, for its tail.
  bf16* panel = nullptr;
  HeadCopy tail = {};
  int chunks_per_pass = units.chunks;
  if (!needs_panel(a->shape)) {
    lent = nullptr;
  } else {
    if (lent) {
      panel = lent;
    } else if (a->logits_cache ? both_in_place(a->shape) : forward_in_place(a->shape)) {
      char* place = a->logits_cache ? static_cast<char*>(a->logits_cache) + logits_bytes(a->shape)
                                    : ws_bytes - L.base >= panel_tile_bytes(a->shape) ? ws + L.base : nullptr;
      if (place) {
        p.head = tail_view(p, reinterpret_cast<const bf16*>(place), kGemmTile);
        tail = tail_copy(p.head);
      }
    } else if (a->logits_cache) {
      panel = reinterpret_cast<bf16*>(static_cast<char*>(a->logits_cache) + logits_bytes(a->shape));
    } else {
      const size_t fit = ws_bytes >= L.total ? (size_t)units.chunks : (ws_bytes - L.base) / (panel_tile_bytes(a->shape) * step_tiles);
      if (fit) panel = reinterpret_cast<bf16*>(ws + L.base);
      if (fit) chunks_per_pass = (int)(fit * step_chunks < (size_t)units.chunks ? fit * step_chunks : (size_t)units.chunks);
    }
  }
  const bool guarded = !p.hidden_aligned || (!panel && !tail.tail && !(is_aligned16(head) && p.V % 8 == 0));
  const GemmLoads loads = guarded ? kGuarded : tail.tail ? kThrough : kCopies;
  for (int chunk0 = 0; chunk0 < units.chunks; chunk0 += chunks_per_pass) {
    const int pass_chunks = min(chunks_per_pass, units.chunks - chunk0);
    HeadCopy copy = tail;
    if (panel) {
      const int tile0 = chunk0 / step_chunks * step_tiles;
      const int pass_tiles = min((pass_chunks + step_chunks - 1) / step_chunks * step_tiles, vocab_tile_count(p.V) - tile0);
      if (!lent || !filled) copy = panel_copy(head, panel, tile0, pass_tiles);
      p.head = panel_view(panel, tile0, pass_tiles);
    }
    const int list_blocks = chunk0 == 0 ? (p.N + 1023) / 1024 : 0;
    if ((rc = launch_prepare<false>(stream, p, CutceRowWork{}, copy, list_blocks, list_blocks == 0))) return rc;
    const auto launch = units.tile == kGemmTile ? launch_stats<4, 4> : launch_stats<2, 4>;
    if ((rc = launch(fn, stream, p, loads, part, chunk0, pass_chunks, units.per_chunk, static_cast<float*>(a->logits_cache))))
      return rc;
  }

  const int merge_blocks = p.n_pad / kMergeSlots;
  LaunchScope scope3("cutce_merge_kernel", stream);
  const bool short_merge = units.chunks <= kShortMerge;
  hipLaunchKernelGGL((short_merge ? cutce_merge_kernel<8> : cutce_merge_kernel<32>), dim3(merge_blocks),
                     dim3(kMergeSlots * (short_merge ? 8 : 32)), 0, stream, p, part, units.chunks, a->lse, sums, a->nll_sum,
                     a->weight_sum);
  return scope3.done();
}

extern "C" int32_t ct_cutce_fwd(void* stream, const ct_cutce_fwd_args* a) {
  CT_REQUIRE(a, "ct_cutce_fwd: null args");
  return cutce_fwd_on(stream, a, a->workspace, a->workspace_bytes, "ct_cutce_fwd");
}

// ---------------------------------------------------------------------------
// The forward for callers that cannot allocate: its workspace (header, active-row
// index list, per-chunk row statistics, per-block loss sums) lives in a static
// device array instead of a caller buffer. Every GPU that loads the library holds
// its own copy of the array at its own address, so the address is looked up once
// per device, with that device current, and kept.
// ---------------------------------------------------------------------------
namespace ct {
constexpr size_t kNoAllocScratchBytes = (size_t)32 << 20;
constexpr int kNoAllocMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
static void* g_scratch_ptr[kNoAllocMaxDevices];  // device address of `scratch`, per device
static std::mutex g_scratch_mutex;
}  // namespace ct

extern "C" size_t ct_cutce_fwd_noalloc_max_bytes(void) { return kNoAllocScratchBytes; }

extern "C" int32_t ct_cutce_fwd_noalloc(void* stream, const ct_cutce_fwd_args* a) {
  CT_REQUIRE(a, "ct_cutce_fwd_noalloc: null args");
  int rc = validate_cutce("ct_cutce_fwd_noalloc", a->shape);
  if (rc) return rc;
  const size_t need = fwd_layout(a->shape).base;  // (a panel, if one is needed, takes what is left)
  if (need > kNoAllocScratchBytes)
    return fail(CT_UNSUPPORTED,
                "ct_cutce_fwd_noalloc: rows=%d, vocab=%d need %zu bytes of scratch, the static "
                "array holds %zu; use ct_cutce_fwd with a caller workspace",
                a->shape.rows, a->shape.vocab, need, kNoAllocScratchBytes);
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess)
    return fail(CT_LAUNCH_FAILED, "ct_cutce_fwd_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  CT_REQUIRE(device >= 0 && device < kNoAllocMaxDevices, "ct_cutce_fwd_noalloc: device %d out of range",
             device);
  void* ws = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
      void* ptr = nullptr;
      e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !ptr)
        return fail(CT_LAUNCH_FAILED, "ct_cutce_fwd_noalloc: hipGetSymbolAddress: %s",
                    hipGetErrorString(e));
      g_scratch_ptr[device] = ptr;
    }
    ws = g_scratch_ptr[device];
  }
  return cutce_fwd_on(stream, a, ws, kNoAllocScratchBytes, "ct_cutce_fwd_noalloc");
}

extern "C" size_t ct_cutce_panel_bytes(const ct_cutce_shape* shape) {
  return valid_sizes(shape) ? full_panel_bytes(*shape) : 0;
}

extern "C" int32_t ct_cutce_head_in_place(const ct_cutce_shape* shape) {
  return valid_sizes(shape) && both_in_place(*shape);
}

extern "C" int32_t ct_cutce_fwd_panel(void* stream, const ct_cutce_fwd_args* a, uint16_t* panel, size_t panel_bytes,
                                      int32_t filled) {
  CT_REQUIRE(a, "ct_cutce_fwd: null args");
  return cutce_fwd_on(stream, a, a->workspace, a->workspace_bytes, "ct_cutce_fwd", reinterpret_cast<bf16*>(panel), panel_bytes,
                      filled != 0);
}

extern "C" int32_t ct_cutce_bwd(void* stream, const ct_cutce_bwd_args* a) { return ct_cutce_bwd_panel(stream, a, nullptr, 0); }

extern "C" int32_t ct_cutce_bwd_panel(void* stream_, const ct_cutce_bwd_args* a, const uint16_t* lent, size_t lent_bytes) {
  CT_REQUIRE(a, "ct_cutce_bwd: null args");
  CT_REQUIRE(a->hidden && a->head && a->targets && a->weights && a->lse && a->dy && a->dhidden &&
                 a->workspace,
             "ct_cutce_bwd: null pointer");
  int rc = validate_cutce("ct_cutce_bwd", a->shape);
  if (!rc) rc = validate_cutce_strides("ct_cutce_bwd", a->shape, a->dhead != nullptr);
  if (rc) return rc;
  CT_REQUIRE(is_aligned16(a->workspace) && is_aligned16(a->dhidden),
             "ct_cutce_bwd: workspace and dhidden must be 16-byte aligned");
  if ((rc = validate_lent("ct_cutce_bwd", a->shape, lent, lent_bytes, a->logits_cache, a->logits_cache_bytes))) return rc;
  const BwdLayout L = bwd_layout(a->shape, a->workspace_bytes, lent || a->logits_cache, a->dhead != nullptr);
  if (L.slab_cols == 0)
    return fail(CT_WORKSPACE_TOO_SMALL, "ct_cutce_bwd: workspace %zu < %zu bytes",
                a->workspace_bytes, ct_cutce_bwd_workspace_min_bytes(&a->shape));
  hipStream_t stream = (hipStream_t)stream_;
  char* ws = static_cast<char*>(a->workspace);
  CutceParams p = make_params(a->hidden, a->head, a->targets, a->weights, a->shape, a->sparse_compaction, ws);
  bf16* G = reinterpret_cast<bf16*>(ws + L.g);
  float* dh_acc = L.slabs > 1 ? reinterpret_cast<float*>(ws + L.acc) : nullptr;
  bf16* dhidden = reinterpret_cast<bf16*>(a->dhidden);
  bf16* dhead = reinterpret_cast<bf16*>(a->dhead);
  const float* cache = static_cast<const float*>(a->logits_cache);
  const int row_blocks = p.n_pad / kGemmTile;
  const size_t params_stride = align_up((size_t)p.n_pad * sizeof(int), 256);
  CutceRowParams rp;
  rp.fac = reinterpret_cast<float*>(ws + L.rowparams);
  rp.lse2 = reinterpret_cast<float*>(ws + L.rowparams + params_stride);
  rp.tgt = reinterpret_cast<int*>(ws + L.rowparams + 2 * params_stride);
  bf16* packed = dhead ? reinterpret_cast<bf16*>(ws + L.packed) : nullptr;
  const bool head_aligned = is_aligned16(a->head) && p.V % 8 == 0;
  const CutceRowWork work = {a->lse, a->dy, rp, packed, dhidden};

  const int cus = device_cu_count();
  const int tiles = vocab_tile_count(p.V);
  const int tiles_per_slab = L.slab_cols / kGemmTile;
  const bf16* head = p.head.base;
  bf16* panel = nullptr;
  HeadCopy tail = {};
  const bool in_place = !lent && (cache ? both_in_place(a->shape) : backward_in_place(a->shape));
  if (head_aligned && p.V % 128) {
    p.head = tail_view(p, reinterpret_cast<const bf16*>(ws + L.tail), 128);
    tail = tail_copy(p.head);
  } else if (needs_panel(a->shape)) {
    // (the forward left panel or tail in the cache)
    const bf16* left = cache ? reinterpret_cast<const bf16*>(reinterpret_cast<const char*>(cache) + logits_bytes(a->shape)) : nullptr;
    if (lent) {
      p.head = panel_view(reinterpret_cast<const bf16*>(lent), 0, tiles);
    } else if (in_place) {
      p.head = tail_view(p, left ? left : reinterpret_cast<const bf16*>(ws + L.panel), kGemmTile);
      if (!left) tail = tail_copy(p.head);
    } else if (left) {
      p.head = panel_view(left, 0, tiles);
    } else {
      panel = reinterpret_cast<bf16*>(ws + L.panel);
    }
  }
  // (an unaligned head with a multiple of 8 columns has no panel)
  const bool guarded_head = !needs_panel(a->shape) && !head_aligned;
  const GemmLoads head_loads = guarded_head ? kGuarded : in_place ? kThrough : kCopies;
  const GemmLoads logits_loads = p.hidden_aligned ? head_loads : kGuarded;
  for (int s = 0; s < L.slabs; ++s) {
    const int slab0 = s * L.slab_cols;
    const int slab_tiles = min(tiles_per_slab, tiles - s * tiles_per_slab);
    const int slab_width = slab_tiles * kGemmTile;
    HeadCopy copy = {};
    if (panel) {
      copy = panel_copy(head, panel, s * tiles_per_slab, slab_tiles);
      p.head = panel_view(panel, s * tiles_per_slab, slab_tiles);
    } else if (s == 0) {
      copy = tail;
    }
    const int per_group = rows_per_group(p.N, p.d), list_blocks = s == 0 ? (p.N + per_group - 1) / per_group : 0;
    if ((list_blocks || panel) && (rc = launch_prepare<true>(stream, p, work, copy, list_blocks, false))) return rc;
    if (cache) {
      LaunchScope scope11("cutce_dlogits_cached_kernel", stream);
      const long threads = (long)(slab_width / kDlogitsRows) * (p.n_pad / 8);
      hipLaunchKernelGGL(cutce_dlogits_cached_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, p, rp,
                         cache, slab0, slab_width, G);
      if ((rc = scope11.done())) return rc;
    } else {
      if (projection_tile(p.N, slab_tiles) == kGemmTile) {
        rc = launch_dlogits<4>("ct_cutce_bwd", stream, p, rp, logits_loads, slab0, slab_tiles,
                               tiles_per_chunk(slab_tiles, row_blocks), G);
      } else {  // (an unpadded head has no columns past the vocabulary to read)
        const int columns = p.head.padded ? slab_width : min(slab_width, p.V - slab0);
        rc = launch_dlogits<2>("ct_cutce_bwd", stream, p, rp, logits_loads, slab0, (columns + 127) / 128, 1, G);
      }
      if (rc) return rc;
    }
    const int mode = L.slabs == 1 ? 0 : (s == 0 ? 1 : (s == L.slabs - 1 ? 3 : 2));
    const CutceSlab slab = {G, packed, slab0, slab_width, mode, dh_acc, dhidden, dhead};
    CutceSplits sp;
    sp.hidden_sums = reinterpret_cast<float*>(ws + L.hidden_sums);
    sp.head_sums = reinterpret_cast<float*>(ws + L.head_sums);
    sp.hidden_room = L.hidden_sums_bytes / sizeof(float);
    sp.head_most = L.head_most;
    // (a slab of a bounded workspace is a short problem whatever the vocabulary: 496 x 640 x 30116 in chunks of 22 rows
    // 1100 -> 722 us, 9540 x 512 x 7604 in chunks of 40 2616 -> 1913; dHead's parts go by the whole vocabulary's tile)
    sp.tile = gradient_tile(ct_cutce_shape{a->shape.rows, a->shape.hidden, slab_width});
    sp.head_tile = gradient_tile(a->shape);
    sp.vocab = tiles * kGemmTile;
    sp.with_head = dhead != nullptr;
    rc = (sp.tile == kGemmTile ? launch_grads<4> : launch_grads<2>)("ct_cutce_bwd", stream, p, slab, sp, head_loads);
    if (rc) return rc;
    if (sp.hidden_room || sp.head_most > 1) {
      LaunchScope scope9("cutce_reduce_kernel", stream);
      const long quads = max((long)p.n_pad * p.d, sp.head_most > 1 ? (long)p.d * slab_width : 0) / 4;
      hipLaunchKernelGGL(cutce_reduce_kernel, dim3((unsigned)min((quads + 255) / 256, (long)cus * 8)), dim3(256), 0, stream, p,
                         slab, sp);
      if ((rc = scope9.done())) return rc;
    }
  }
  return CT_OK;
}
