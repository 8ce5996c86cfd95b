// Workgroup-tile bf16 GEMM core for gfx950, used by the cut cross-entropy kernels.
//
// 4 wavefronts in a 2 x 2 arrangement, each with NB x NB mfma32 accumulator blocks. NB = 4: a tile of
// 256 x 256, 256 f32 registers per lane, one workgroup per compute unit; NB = 2: 128 x 128, 64 registers, two
// workgroups per compute unit, for problems with few tiles (which one: projection_tile and gradient_tile in
// ct_cutce.hip). The contraction runs in steps of BK = 32.
//
// An operand comes in one of two memory layouts:
//   KcLoader  "k-contiguous": matrix rows are the M (or N) index, the
//             contraction index is contiguous. LDS tile [64 NB][2 BK], two steps, MFMA
//             fragments read with ds_read_b128 (KcStepLoader: one step, for the guarded loop).
//   McLoader  "m-contiguous": matrix rows are the contraction index, the M
//             (or N) index is contiguous. LDS tile [BK][64 NB], fragments read
//             with transposed LDS reads.
// The rows of a k-contiguous operand can be addressed through an index list (gather).
//
// Three main loops share the loaders; a kernel is compiled for one of them (GemmLoads), because more than one in
// a kernel cost it registers, spills and instruction cache:
//   pipelined  operands 16-byte aligned, contraction a multiple of 128: tiles are copied global ->
//              LDS asynchronously, three steps ahead, into a ring of 4 LDS stages; MFMA fragments
//              are double buffered in registers so that LDS reads of the next half step overlap
//              the current MFMAs; one barrier per step (gen_gemm_asm.py). Rows or
//              columns of a tile past the end of the matrix are copies of valid ones.
//   through registers  the same loop where the rows of one operand start at any multiple of 2 bytes and the tile
//              lies inside of the matrix: that operand's chunks are loaded into registers two to three steps ahead
//              and stored to the LDS ring one step ahead (unaligned global loads; the copies need aligned chunks).
//   guarded    unaligned operands: element-wise guarded loads that zero fill, staged through
//              registers, 2 LDS stages.
#pragma once

#include <type_traits>

#include "ct_common.hip.h"
#include "ct_gemm_asm.inc"

namespace ct {

constexpr int kGemmTile = 256;  // of the large tile, and what row blocks and vocabulary are padded to
constexpr int kGemmBK = 32;

enum class GemmLoads { kCopies, kThroughRegisters, kGuarded };

CT_DEVICE u32x4 load_chunk_guarded(const bf16* p, int count) {
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = e < count ? p[e] : (bf16)0.f;
  return as_u32x4(v);
}

// A workgroup's tile: 4 wavefronts of NB x NB accumulator blocks. RING: stages of A (8: the small tile for launches of
// no more workgroups than compute units, whose copies nothing but their own number hides).
template <int NB, int RING = 4>
struct GemmShape {
  static constexpr int kTile = 64 * NB, kWave = 32 * NB;
  static constexpr int kTileBytes = kTile * kGemmBK * 2;  // NB = 4: 16 KB
  static constexpr int kStageBytes = 2 * kTileBytes;      // of the guarded loop: A tile then B tile
  static constexpr int kStages = RING;
  // of the others: RING stages of A, a step each, then half as many of B, two steps each
  static constexpr int kB = kStages * kTileBytes, kPairBytes = 2 * kTileBytes;
  static constexpr int kGroups = NB == 4 || RING == 8 ? 1 : 2;         // workgroups per compute unit that registers are for
  static constexpr size_t kBytes = (size_t)kStages * kStageBytes;  // NB = 4: 128 KB
};

// In all loaders thread t owns the 16-byte LDS slots t + 256 n of the tile: slot P holds physical chunk P % CPR of
// row P / CPR, i.e. logical chunk (P % CPR) ^ swizzle(row); voff[n] is the byte offset of that chunk from `base` at
// k = 0 (32 bits: the host checks sizes and strides against it).
template <int NB, int STEPS>
struct KcRows {
  static constexpr int CPR = STEPS * kGemmBK / 8;  // 4 a step
  static constexpr int NCH = NB * STEPS;
  static constexpr int kRowsPerPass = 256 / CPR;
  const char* base;    // uniform
  unsigned voff[NCH];
  int chunk;

  // rows m0 .. of `base_` (leading dimension ld elements), optionally
  // gathered through row_index. Rows >= rows_valid are copies of the first row (callers discard
  // what they get from them).
  // With interleave_rows, row 32 nb + j of a wavefront's rows holds matrix row NB j + nb of them:
  // in the accumulator layout lane j of a wavefront then owns NB consecutive matrix rows (its
  // column blocks), which an epilogue can store with one access.
  CT_DEVICE void init_rows(const bf16* base_, long ld, const int* row_index, int m0, int rows_valid, bool interleave_rows) {
    const int t = threadIdx.x;
    const bool gathered = row_index != nullptr;
    base = reinterpret_cast<const char*>(gathered ? base_ : base_ + (size_t)m0 * ld);
    const int r0 = t / CPR;
    chunk = (t % CPR) ^ swizzle<CPR>(r0);  // rows r0 + kRowsPerPass n share the swizzle
    int src[NCH];
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      const int tile_row = r0 + kRowsPerPass * n;
      constexpr int wave_rows = 32 * NB;
      const int r = interleave_rows ? ((tile_row & wave_rows) | ((tile_row & 31) * NB) | ((tile_row >> 5) % NB)) : tile_row;
      const bool ok = m0 + r < rows_valid;
      src[n] = gathered ? (ok ? m0 + r : 0) : (ok ? r : 0);
    }
    if (gathered) {  // (one branch around all of the loads: they travel together)
#pragma unroll
      for (int n = 0; n < NCH; ++n) src[n] = row_index[src[n]];
    }
#pragma unroll
    for (int n = 0; n < NCH; ++n) voff[n] = (unsigned)(((long)src[n] * ld + chunk * 8) * 2);
  }
};

template <int NB>
struct KcLoader : KcRows<NB, 2> {
  typedef KcRows<NB, 2> Rows;
  typedef RowFragOffsets<Rows::CPR> FragOffsets;
  CT_DEVICE void init(const bf16* base_, long ld, const int* row_index, int m0, int rows_valid, int, bool interleave_rows = false) {
    this->init_rows(base_, ld, row_index, m0, rows_valid, interleave_rows);
  }
  // copies of the steps at k0 and behind
  CT_DEVICE void dma(int k0, lds_addr tile) const {
    const int wave = uniform(threadIdx.x >> 6);
    const char* p = this->base + (size_t)k0 * 2;
#pragma unroll
    for (int n = 0; n < Rows::NCH; ++n) dma16_s(p, this->voff[n], tile + (n * 256 + wave * 64) * 16);
  }
};

// One step at a time, by loads that read k >= k_valid as zero.
template <int NB>
struct KcStepLoader : KcRows<NB, 1> {
  static constexpr int NCH = NB, CPR = KcRows<NB, 1>::CPR;
  u32x4 regs[NCH];
  int k_valid;
  CT_DEVICE void init(const bf16* base_, long ld, const int* row_index, int m0, int rows_valid,
                      int k_valid_, bool interleave_rows = false) {
    k_valid = k_valid_;
    this->init_rows(base_, ld, row_index, m0, rows_valid, interleave_rows);
  }
  CT_DEVICE void fetch(int k0) {
    const int k = k0 + this->chunk * 8;
    const int count = min(max(k_valid - k, 0), 8);
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      regs[n] = count ? load_chunk_guarded(reinterpret_cast<const bf16*>(this->base + (size_t)k0 * 2 + this->voff[n]), count)
                      : u32x4{0u, 0u, 0u, 0u};
    }
  }
  CT_DEVICE void commit(lds_addr tile) const {
#pragma unroll
    for (int n = 0; n < NCH; ++n) lds_store<u32x4>(tile + (n * 256 + (int)threadIdx.x) * 16, regs[n]);
  }
  // fragment for the wavefront's 32-row block i, contraction steps 16*ks .. 16*ks+15;
  // `wave_first` (multiple of 128) is the wavefront's first row.
  typedef RowFragOffsets<CPR> FragOffsets;
  static CT_DEVICE bf16x8 frag(int tile_off, const FragOffsets& fo, int ks, int wave_first, int i) {
    return fo.load(tile_off + (wave_first / 32) * FragOffsets::kRowBlockBytes, i, ks);
  }
};

template <int NB>
struct McLoader {
  static constexpr int CPR = 8 * NB;           // 16-byte chunks of a tile row
  static constexpr int NCH = NB;
  static constexpr int kRowsPerPass = 256 / CPR;
  const char* base;  // uniform: column m0 of row 0
  long ld;
  unsigned voff[NCH];
  u32x4 regs[NCH];
  int col[2];  // first column of the chunk fetched in even / odd passes
  int cols_left, k_valid;

  // columns m0 .. of `base_`. The guarded loop reads columns >= cols_valid and rows >= k_valid
  // as zero; the pipelined one, where cols_valid is a multiple of 8, such columns as copies of the
  // tile's first 8 (callers discard what they get from them).
  CT_DEVICE void init(const bf16* base_, long ld_, int m0, int cols_valid, int k_valid_) {
    const int t = threadIdx.x;
    base = reinterpret_cast<const char*>(base_ + m0);
    ld = ld_;
    k_valid = k_valid_;
    cols_left = cols_valid - m0;
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      const int r = t / CPR + kRowsPerPass * n;
      int c = ((t % CPR) ^ swizzle<CPR>(r)) * 8;
      col[n & 1] = c;
      if (c >= cols_left) c = 0;
      voff[n] = (unsigned)(((long)r * ld + c) * 2);
    }
  }
  CT_DEVICE void dma(int k0, lds_addr tile) const {
    const int wave = uniform(threadIdx.x >> 6);
    const char* p = base + (size_t)k0 * ld * 2;
#pragma unroll
    for (int n = 0; n < NCH; ++n) dma16_s(p, voff[n], tile + (n * 256 + wave * 64) * 16);
  }
  CT_DEVICE void fetch(int k0) {
    const int r0 = (int)threadIdx.x / CPR;
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      const int k = k0 + r0 + kRowsPerPass * n;
      const int count = min(max(cols_left - col[n & 1], 0), 8);
      if (k < k_valid && count) {
        regs[n] = load_chunk_guarded(reinterpret_cast<const bf16*>(base + (size_t)k0 * ld * 2 + voff[n]), count);
      } else {
        regs[n] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  }
  CT_DEVICE void commit(lds_addr tile) const {
#pragma unroll
    for (int n = 0; n < NCH; ++n) lds_store<u32x4>(tile + (n * 256 + (int)threadIdx.x) * 16, regs[n]);
  }
  typedef TrFragOffsets<CPR, KSlots::kNatural> FragOffsets;
  static CT_DEVICE bf16x8 frag(int tile_off, const FragOffsets& fo, int ks, int wave_first, int i) {
    return fo.load(tile_off + (wave_first / 128) * 256, ks, i);
  }
};

template <int NB, GemmLoads LOADS>
using GemmB = std::conditional_t<LOADS == GemmLoads::kGuarded, KcStepLoader<NB>, KcLoader<NB>>;

template <int NB>
struct GemmAcc {
  typedef float Lane __attribute__((ext_vector_type(NB)));  // a lane's consecutive elements of a row
  f32x16 c[NB][NB];
  CT_DEVICE void clear() {
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b) c[a][b] = zero16();
  }
  // Wait states between the compiler's last MFMA and value(), whose read it does not see.
  CT_DEVICE void settle() {
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b) asm volatile("" : "+a"(c[a][b]));
    asm volatile("s_nop 15\n\ts_nop 7");
  }
  // An element, read where the call stands. (An epilogue's branches otherwise have the reads and what
  // is computed from them moved in front of the branch, where 256 of them do not fit and spill.)
  CT_DEVICE float value(int i, int nb, int r) const {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(c[i][nb][r]));
    return v;
  }
  CT_DEVICE Lane lane(int i, int r) const {
    Lane out;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) out[nb] = value(i, nb, r);
    return out;
  }
};

// Stores of a lane's consecutive elements at a wave-uniform address plus a 32-bit lane offset.
CT_DEVICE void store_lane(void* row, unsigned lane_offset, f32x4 v) { store_global16_s<0>(row, lane_offset, v); }
CT_DEVICE void store_lane(void* row, unsigned lane_offset, bf16x4 v) { store_global8_s<0>(row, lane_offset, v); }
CT_DEVICE void store_lane(void* row, unsigned lane_offset, f32x2 v) {
  store_global8_s<0>(row, lane_offset, __builtin_bit_cast(bf16x4, v));
}
CT_DEVICE void store_lane(void* row, unsigned lane_offset, bf16x2 v) {
  store_global4_s<0>(row, lane_offset, __builtin_bit_cast(float, v));
}
CT_DEVICE bf16x4 to_bf16(f32x4 v) { return bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]}; }
CT_DEVICE bf16x2 to_bf16(f32x2 v) { return bf16x2{(bf16)v[0], (bf16)v[1]}; }

struct GemmFrags {
  bf16x8 a[4], b[4];
};

CT_DEVICE void load_frags(GemmFrags& f, int stage_off, const McLoader<4>::FragOffsets& afo,
                          const KcStepLoader<4>::FragOffsets& bfo, int ks, int wm, int wn) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f.a[i] = McLoader<4>::frag(stage_off, afo, ks, wm, i);
    f.b[i] = KcStepLoader<4>::frag(stage_off + GemmShape<4>::kTileBytes, bfo, ks, wn, i);
  }
}

CT_DEVICE void mfma_block(const GemmFrags& f, GemmAcc<4>& acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int jn = 0; jn < 4; ++jn) acc.c[i][jn] = mfma32(f.a[i], f.b[jn], acc.c[i][jn]);
}

// s_waitcnt vmcnt(16) (expcnt / lgkmcnt left at "no wait")
CT_DEVICE void wait_vmcnt16() { __builtin_amdgcn_s_waitcnt(0x0F70 | (1 << 14)); }
// Execution barrier without the memory fence of __syncthreads() (which would wait for
// every copy in flight); callers order their own LDS traffic with the waits above.
CT_DEVICE void workgroup_barrier() { __builtin_amdgcn_s_barrier(); }

// The pipelined main loop with a fixed instruction order (see gen_gemm_asm.py), for an
// m-contiguous A, a k-contiguous B and a step count that is a positive multiple of 4. Entered with A's copies of steps 0..2
// and B's of pairs 0 and 1 issued, those of step 0 landed for every wavefront; returns with nothing in flight and the LDS tiles free. It adds to the accumulators (kAdd) or writes them
// (kFresh; kFreshBehindStores: at least kStoresBehindCopies stores of every wavefront follow these copies, or they
// have landed).
enum class GemmStart { kAdd, kFresh, kFreshBehindStores };
CT_DEVICE unsigned long long uniform64(const void* p) {
  const unsigned long long b = (unsigned long long)(uintptr_t)p;
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
  return ((unsigned long long)hi << 32) | (unsigned long long)lo;
}
// Operands of the loops' asm statements. THROUGH: the operand that comes through registers (A: CT_GEMM_VIA_A_LOOP, from C = 0;
// B: CT_GEMM_VIA_B_LOOP, adding), entered with the other one's copies issued and none of its own loads.
enum class Through { kNone, kA, kB };
// Where the source of B's copies starts: at the pair behind those that a loop is entered with, or at the last pair.
template <int RING = 4>
CT_DEVICE int first_pair(int k_begin, int steps) { return k_begin + min(RING, steps - 2) * kGemmBK; }
template <GemmStart START, Through THROUGH = Through::kNone>
CT_DEVICE void gemm_loop_scheduled(const McLoader<4>& A, const KcLoader<4>& B, int k_begin, int steps,
                                   lds_addr smem, const McLoader<4>::FragOffsets& afo,
                                   const KcLoader<4>::FragOffsets& bfo, int wm, int wn, GemmAcc<4>& acc) {
  const int wave = uniform(threadIdx.x >> 6);
  // sources of the copies of step 3, of the loads of step 0
  const int first_a = k_begin + (THROUGH == Through::kA ? 0 : 3 * kGemmBK);
  const int first_b = THROUGH == Through::kB ? k_begin : first_pair(k_begin, steps);
  const unsigned long long src_a = uniform64(A.base + (size_t)first_a * (size_t)A.ld * 2);
  const unsigned long long src_b = uniform64(B.base + (size_t)first_b * 2);
  const unsigned stride_a = (unsigned)uniform((int)(kGemmBK * A.ld * 2));
  const unsigned steps_u = (unsigned)uniform(steps);
  const unsigned lds_wave = (unsigned)uniform((int)(uintptr_t)(smem + wave * 1024));
  const int a_off = (wm / 128) * 256;
  const int b_off = GemmShape<4>::kB + (wn / 32) * KcLoader<4>::FragOffsets::kRowBlockBytes;
#define CT_GEMM_ACC(mode) \
  mode(acc.c[0][0]), mode(acc.c[0][1]), mode(acc.c[0][2]), mode(acc.c[0][3]), mode(acc.c[1][0]), mode(acc.c[1][1]), mode(acc.c[1][2]), mode(acc.c[1][3]), \
      mode(acc.c[2][0]), mode(acc.c[2][1]), mode(acc.c[2][2]), mode(acc.c[2][3]), mode(acc.c[3][0]), mode(acc.c[3][1]), mode(acc.c[3][2]), mode(acc.c[3][3])
#define CT_GEMM_IN \
  "s"(src_a), "s"(src_b), "s"(stride_a), "s"(steps_u), "s"(lds_wave), "v"(afo.ptr[0][0] + a_off), \
      "v"(afo.ptr[0][1] + a_off), "v"(afo.ptr[0][2] + a_off), "v"(afo.ptr[0][3] + a_off), "v"(afo.ptr[1][0] + a_off), \
      "v"(afo.ptr[1][1] + a_off), "v"(afo.ptr[1][2] + a_off), "v"(afo.ptr[1][3] + a_off), "v"(bfo.ptr[0] + b_off), \
      "v"(bfo.ptr[1] + b_off), "v"(bfo.ptr[2] + b_off), "v"(bfo.ptr[3] + b_off), "v"(A.voff[0]), "v"(A.voff[1]), \
      "v"(A.voff[2]), "v"(A.voff[3]), "v"(B.voff[0]), "v"(B.voff[1]), "v"(B.voff[2]), "v"(B.voff[3]), "v"(B.voff[4]), \
      "v"(B.voff[5]), "v"(B.voff[6]), "v"(B.voff[7])
  if constexpr (THROUGH != Through::kNone) {
    static_assert((THROUGH == Through::kA) == (START != GemmStart::kAdd), "the forms that there are");
    const lds_addr thread = smem + (THROUGH == Through::kB ? GemmShape<4>::kB : 0) + (int)threadIdx.x * 16;
    if constexpr (THROUGH == Through::kA)
      asm volatile(CT_GEMM_VIA_A_LOOP : CT_GEMM_ACC("=&a") : CT_GEMM_IN, "v"(thread)
                   : "memory", "m0", "scc", CT_GEMM_VIA_LOOP_CLOBBERS);
    else
      asm volatile(CT_GEMM_VIA_B_LOOP : CT_GEMM_ACC("+a") : CT_GEMM_IN, "v"(thread)
                   : "memory", "m0", "scc", CT_GEMM_VIA_LOOP_CLOBBERS);
  } else if constexpr (START == GemmStart::kAdd)
    asm volatile(CT_GEMM_LOOP : CT_GEMM_ACC("+a") : CT_GEMM_IN : "memory", "m0", "scc", CT_GEMM_LOOP_CLOBBERS);
  else if constexpr (START == GemmStart::kFresh)
    asm volatile(CT_GEMM_FRESH_LOOP : CT_GEMM_ACC("=&a") : CT_GEMM_IN : "memory", "m0", "scc", CT_GEMM_LOOP_CLOBBERS);
  else
    asm volatile(CT_GEMM_FRESH_LOOP_BEHIND_STORES : CT_GEMM_ACC("=&a") : CT_GEMM_IN
                 : "memory", "m0", "scc", CT_GEMM_LOOP_CLOBBERS);
#undef CT_GEMM_ACC
#undef CT_GEMM_IN
}

// The copies that a loop is entered with: A's of steps STEP .. END - 1, B's of a pair.
template <int STEP, int END, int NB>
CT_DEVICE void copy_steps(const McLoader<NB>& A, int k_begin, lds_addr smem) {
#pragma unroll
  for (int i = STEP; i < END; ++i) A.dma(k_begin + i * kGemmBK, smem + i * GemmShape<NB>::kTileBytes);
}
template <int RING, int NB>
CT_DEVICE void copy_pair_at(const KcLoader<NB>& B, int stage, int k0, lds_addr smem) {
  B.dma(k0, smem + GemmShape<NB, RING>::kB + stage * GemmShape<NB, RING>::kPairBytes);
}
template <int NB>
CT_DEVICE void copy_pair(const KcLoader<NB>& B, int pair, int k_begin, lds_addr smem) {
  copy_pair_at<4>(B, pair, k_begin + pair * 2 * kGemmBK, smem);
}
// Those of step 0 first, then the rest: `behind step 0` many.
constexpr int kCopiesBehindStep0 = 4 + 4 + 8;
CT_DEVICE void gemm_copy_ahead(const McLoader<4>& A, const KcLoader<4>& B, int k_begin, lds_addr smem) {
  copy_steps<0, 1>(A, k_begin, smem);
  copy_pair(B, 0, k_begin, smem);
  copy_steps<1, 3>(A, k_begin, smem);
  copy_pair(B, 1, k_begin, smem);
}

// acc = A[m-tile, 0:k_end] * B[n-tile, 0:k_end]^T behind gemm_copy_ahead, k_end a positive multiple of 128. STORES:
// every wavefront has issued at least kStoresBehindCopies stores since, or it waits for all of the copies (`landed`).
constexpr int kStoresBehindCopies = 55;  // what the waits of CT_GEMM_FRESH_LOOP_BEHIND_STORES need (gen_gemm_asm.py)
template <bool STORES>
CT_DEVICE void gemm_tile_fresh(const McLoader<4>& A, const KcLoader<4>& B, int k_end, lds_addr smem, GemmAcc<4>& acc, bool landed) {
  constexpr GemmStart kStart = STORES ? GemmStart::kFreshBehindStores : GemmStart::kFresh;
  const int w = threadIdx.x >> 6;
  const McLoader<4>::FragOffsets afo(smem);
  const KcLoader<4>::FragOffsets bfo(smem);
  // step 0's copies: at least 16 + 55 others behind them, or the 16 of the other steps
  if (!STORES) wait_vmcnt16();
  else if (landed) dma_wait_all();
  else asm volatile("s_waitcnt vmcnt(63)" ::: "memory");
  workgroup_barrier();
  gemm_loop_scheduled<kStart>(A, B, 0, k_end / kGemmBK, smem, afo, bfo, (w >> 1) * 128, (w & 1) * 128, acc);
}

// acc = the same product with A through registers, behind B's two pairs of copies.
CT_DEVICE void gemm_tile_through_a(const McLoader<4>& A, const KcLoader<4>& B, int k_end, lds_addr smem, GemmAcc<4>& acc) {
  const int w = threadIdx.x >> 6;
  const McLoader<4>::FragOffsets afo(smem);
  const KcLoader<4>::FragOffsets bfo(smem);
  gemm_loop_scheduled<GemmStart::kFresh, Through::kA>(A, B, 0, k_end / kGemmBK, smem, afo, bfo, (w >> 1) * 128, (w & 1) * 128, acc);
}

// acc += A[m-tile, k_begin:k_end] * B[n-tile, k_begin:k_end]^T (k_end - k_begin a multiple of 128
// unless kGuarded; kThroughRegisters: B comes through them). Must be called by all 256 threads; ends with the LDS tiles free for reuse.
template <GemmLoads LOADS>
CT_DEVICE void gemm_tile(McLoader<4>& A, GemmB<4, LOADS>& B, int k_begin, int k_end, lds_addr smem, GemmAcc<4>& acc) {
  const int w = threadIdx.x >> 6;
  const int wm = (w >> 1) * 128, wn = (w & 1) * 128;
  if (k_begin >= k_end) return;
  const McLoader<4>::FragOffsets afo(smem);
  const typename GemmB<4, LOADS>::FragOffsets bfo(smem);
  if constexpr (LOADS != GemmLoads::kGuarded) {
    const int steps = (k_end - k_begin) / kGemmBK;
    dma_wait_all();  // nothing of ours may still be in flight when counting copies below
    if constexpr (LOADS == GemmLoads::kCopies) {
      gemm_copy_ahead(A, B, k_begin, smem);
      static_assert(kCopiesBehindStep0 == 16, "the wait leaves the copies behind step 0's in flight");
      wait_vmcnt16();
      workgroup_barrier();
      gemm_loop_scheduled<GemmStart::kAdd>(A, B, k_begin, steps, smem, afo, bfo, wm, wn, acc);
    } else {
      copy_steps<0, 3>(A, k_begin, smem);
      gemm_loop_scheduled<GemmStart::kAdd, Through::kB>(A, B, k_begin, steps, smem, afo, bfo, wm, wn, acc);
    }
  } else {
    constexpr int BK = kGemmBK, kTile = GemmShape<4>::kTileBytes, kStage = GemmShape<4>::kStageBytes;
    A.fetch(k_begin);
    B.fetch(k_begin);
    A.commit(smem);
    B.commit(smem + kTile);
    __syncthreads();
    int cur = 0, nxt = kStage;
    for (int k0 = k_begin; k0 < k_end; k0 += BK) {
      const bool more = k0 + BK < k_end;
      if (more) {
        A.fetch(k0 + BK);
        B.fetch(k0 + BK);
      }
#pragma unroll
      for (int ks = 0; ks < BK / 16; ++ks) {
        GemmFrags f;
        load_frags(f, cur, afo, bfo, ks, wm, wn);
        mfma_block(f, acc);
      }
      if (more) {
        A.commit(smem + nxt);
        B.commit(smem + nxt + kTile);
      }
      __syncthreads();
      const int tmp = cur;
      cur = nxt;
      nxt = tmp;
    }
    acc.settle();
  }
}

// The small tile (NB = 2: 128 x 128, 64 accumulator registers, two workgroups per compute unit), with a fixed order of its
// own (gen_gemm_asm.py).
// This lane's part of the wavefront's fragments of A, stage 0.
struct SmallFrags {
  lds_addr a[2][2];
  CT_DEVICE explicit SmallFrags(lds_addr smem) {
    const int wm = (uniform(threadIdx.x >> 6) >> 1) * GemmShape<2>::kWave, l = lane_id();
#pragma unroll
    for (int second = 0; second < 2; ++second)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 8 * (l >> 5) + 4 * second + ((l & 15) >> 2), col = wm + 32 * i + 16 * ((l >> 4) & 1) + 4 * (l & 3);
        a[second][i] = smem + tile_byte_offset<McLoader<2>::CPR>(row, col >> 3) + (col & 4) * 2;
      }
  }
};
// The row block of B that a wavefront starts at.
CT_DEVICE int small_first_block() { return (uniform(threadIdx.x >> 6) & 1) * 2; }

// acc += the product, entered with A's copies of the first four steps and B's of two pairs issued (those of step 0
// landed for every wavefront, this one's of A's step 1 too), of an operand through registers none.
template <Through THROUGH, int RING = 4>
CT_DEVICE void gemm_small_loop(const McLoader<2>& A, const KcLoader<2>& B, int k_begin, int k_end, lds_addr smem, GemmAcc<2>& acc) {
  const SmallFrags f(smem);
  constexpr int kB = GemmShape<2, RING>::kB;
  const int loop_steps = (k_end - k_begin) / kGemmBK;
  const KcLoader<2>::FragOffsets b(smem + kB + small_first_block() * KcLoader<2>::FragOffsets::kRowBlockBytes);
  const int first_a = k_begin + (THROUGH == Through::kA ? 0 : (RING == 4 ? 3 : min(RING, loop_steps) - 1) * kGemmBK);
  const int first_b = THROUGH == Through::kB ? k_begin : first_pair<RING>(k_begin, loop_steps);
  const unsigned long long src_a = uniform64(A.base + (size_t)first_a * (size_t)A.ld * 2);
  const unsigned long long src_b = uniform64(B.base + (size_t)first_b * 2);
  const unsigned stride_a = (unsigned)uniform((int)(kGemmBK * A.ld * 2));
  const unsigned steps = (unsigned)uniform(loop_steps);
  const unsigned lds_wave = (unsigned)uniform((int)(uintptr_t)(smem + uniform(threadIdx.x >> 6) * 1024));
#define CT_GEMM_SMALL_ACC "+a"(acc.c[0][0]), "+a"(acc.c[0][1]), "+a"(acc.c[1][0]), "+a"(acc.c[1][1])
#define CT_GEMM_SMALL_IN \
  "s"(src_a), "s"(src_b), "s"(stride_a), "s"(steps), "s"(lds_wave), "v"(f.a[0][0]), "v"(f.a[0][1]), "v"(f.a[1][0]), \
      "v"(f.a[1][1]), "v"(b.ptr[0]), "v"(b.ptr[1]), "v"(b.ptr[2]), "v"(b.ptr[3]), "v"(A.voff[0]), "v"(A.voff[1]), \
      "v"(B.voff[0]), "v"(B.voff[1]), "v"(B.voff[2]), "v"(B.voff[3])
  if constexpr (THROUGH == Through::kNone && RING == 8) {
    asm volatile(CT_GEMM_SMALL_DEEP_LOOP : CT_GEMM_SMALL_ACC : CT_GEMM_SMALL_IN
                 : "memory", "m0", "scc", CT_GEMM_SMALL_LOOP_CLOBBERS);
  } else if constexpr (THROUGH == Through::kNone) {
    asm volatile(CT_GEMM_SMALL_LOOP : CT_GEMM_SMALL_ACC : CT_GEMM_SMALL_IN
                 : "memory", "m0", "scc", CT_GEMM_SMALL_LOOP_CLOBBERS);
  } else {
    const lds_addr thread = smem + (THROUGH == Through::kB ? kB : 0) + (int)threadIdx.x * 16;
    if constexpr (RING == 8)
      asm volatile(CT_GEMM_SMALL_DEEP_VIA_A_LOOP : CT_GEMM_SMALL_ACC : CT_GEMM_SMALL_IN, "v"(thread)
                   : "memory", "m0", "scc", CT_GEMM_SMALL_DEEP_VIA_LOOP_CLOBBERS);
    else if constexpr (THROUGH == Through::kA)
      asm volatile(CT_GEMM_SMALL_VIA_A_LOOP : CT_GEMM_SMALL_ACC : CT_GEMM_SMALL_IN, "v"(thread)
                   : "memory", "m0", "scc", CT_GEMM_SMALL_VIA_LOOP_CLOBBERS);
    else
      asm volatile(CT_GEMM_SMALL_VIA_B_LOOP : CT_GEMM_SMALL_ACC : CT_GEMM_SMALL_IN, "v"(thread)
                   : "memory", "m0", "scc", CT_GEMM_SMALL_VIA_LOOP_CLOBBERS);
  }
#undef CT_GEMM_SMALL_ACC
#undef CT_GEMM_SMALL_IN
}

// acc += A[m-tile, k_begin:k_end] * B[n-tile, k_begin:k_end]^T in the small tile; THROUGH: the operand of kThroughRegisters.
template <GemmLoads LOADS, Through THROUGH = Through::kB, int RING = 4>
CT_DEVICE void gemm_tile(McLoader<2>& A, GemmB<2, LOADS>& B, int k_begin, int k_end, lds_addr smem, GemmAcc<2>& acc) {
  if (k_begin >= k_end) return;
  if constexpr (LOADS == GemmLoads::kCopies && RING == 8) {
    // (past the end the last step and pair again: nobody reads them)
    const int last = k_end - kGemmBK, last_pair = k_end - 2 * kGemmBK;
    dma_wait_all();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i % 2) copy_pair_at<8>(B, i / 2, min(k_begin + (i - 1) * kGemmBK, last_pair), smem);
      A.dma(min(k_begin + i * kGemmBK, last), smem + i * GemmShape<2>::kTileBytes);
    }
    // (32 copies, the 6 of step 0 first)
    asm volatile("s_waitcnt vmcnt(26)\n\ts_barrier" ::: "memory");
    gemm_small_loop<Through::kNone, 8>(A, B, k_begin, k_end, smem, acc);
  } else if constexpr (LOADS == GemmLoads::kCopies) {
    dma_wait_all();  // nothing of ours may still be in flight when counting copies below
    copy_steps<0, 1>(A, k_begin, smem);
    copy_pair(B, 0, k_begin, smem);
    copy_steps<1, 2>(A, k_begin, smem);
    copy_pair(B, 1, k_begin, smem);
    copy_steps<2, 4>(A, k_begin, smem);
    // step 0 and A's step 1 have landed
    static_assert(2 * McLoader<2>::NCH + KcLoader<2>::NCH == 8, "the wait leaves A's steps 2 and 3 and a pair in flight");
    asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    gemm_small_loop<Through::kNone>(A, B, k_begin, k_end, smem, acc);
  } else if constexpr (LOADS == GemmLoads::kThroughRegisters) {
    dma_wait_all();
    if constexpr (THROUGH == Through::kA) {
#pragma unroll
      for (int pair = 0; pair < RING / 2; ++pair)
        copy_pair_at<RING>(B, pair, min(k_begin + pair * 2 * kGemmBK, k_end - 2 * kGemmBK), smem);
    } else {
      copy_steps<0, 4>(A, k_begin, smem);
    }
    gemm_small_loop<THROUGH, RING>(A, B, k_begin, k_end, smem, acc);
  } else {
    constexpr int kTile = GemmShape<2>::kTileBytes;
    typedef KcStepLoader<2>::FragOffsets StepOffsets;
    const SmallFrags frags(smem);
    const StepOffsets b_ptr(smem + kTile + small_first_block() * StepOffsets::kRowBlockBytes);
#pragma nounroll
    for (int k0 = k_begin; k0 < k_end; k0 += kGemmBK) {
      A.fetch(k0);
      B.fetch(k0);
      A.commit(smem);
      B.commit(smem + kTile);
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        bf16x8 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int off = ks * (16 * McLoader<2>::CPR * 16);
          const bf16x4_vs lo = lds_load_tr(frags.a[0][i] + off), hi = lds_load_tr(frags.a[1][i] + off);
          a[i] = bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          b[i] = b_ptr.load(0, i, ks);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc.c[i][j] = mfma32(a[i], b[j], acc.c[i][j]);
      }
      __syncthreads();
    }
    acc.settle();
  }
}

// The rows of a wavefront's tile in the order of its accumulators (0..3, 8..11, ...; lanes of the other half
// are 4 rows on), as a scalar address that advances. The stride is opaque: as a loop invariant its
// 64 multiples are formed in front of the persistent loop and spilled.
struct TileRows {
  char* row;
  int stride;  // bytes
  CT_DEVICE TileRows(void* origin, int stride_) : row(reinterpret_cast<char*>(origin)), stride(uniform(stride_)) {
    asm volatile("" : "+s"(stride));
  }
  CT_DEVICE void advance(int r) { row += (long)stride * ((r & 3) == 3 ? 5 : 1); }
};

// The tiles of a kernel one after the other: begin() as soon as a tile's loaders are known (the LDS stages are
// free from the end of the last run() on), run() for its product, store() for the rows that an epilogue writes.
// In the large tile's pipelined form the copies of a tile's first three steps then travel behind the epilogue of
// the tile before: with one workgroup on a compute unit nothing else hides them. What run() waits for goes by the
// stores counted since begin() (a constant wherever an epilogue issues them on every path): where they are too
// few for the counted waits, as on a kernel's first tile, it waits for all copies.
// kThroughRegisters (A): only B's copies travel ahead.
template <int NB, GemmLoads LOADS, bool STORES, int RING = 4>
struct GemmTiles {
  typedef GemmB<NB, LOADS> LoaderB;
  static constexpr bool kAhead = NB == 4 && LOADS == GemmLoads::kCopies;
  int stores = 0;  // of this wavefront behind the copies of begin()
  CT_DEVICE void begin(const McLoader<NB>& A, const LoaderB& B, lds_addr smem) {
    if constexpr (kAhead) {
      gemm_copy_ahead(A, B, 0, smem);
    } else if constexpr (NB == 4 && LOADS == GemmLoads::kThroughRegisters) {
      copy_pair(B, 0, 0, smem);
      copy_pair(B, 1, 0, smem);
    }
  }
  // a lane's NB consecutive elements of accumulator row r of a block (wave-uniform control flow only)
  template <class Elements>
  CT_DEVICE void store(TileRows& rows, unsigned lane_offset, int r, Elements x) {
    static_assert(STORES, "a kernel that stores this way waits by their count");
    store_lane(rows.row, lane_offset, x);
    rows.advance(r);
    if constexpr (kAhead) ++stores;
  }
  CT_DEVICE void run(McLoader<NB>& A, LoaderB& B, int k_end, lds_addr smem, GemmAcc<NB>& acc) {
    if constexpr (kAhead) {
      gemm_tile_fresh<STORES>(A, B, k_end, smem, acc, stores < kStoresBehindCopies);
      stores = 0;
    } else if constexpr (NB == 4 && LOADS == GemmLoads::kThroughRegisters) {
      gemm_tile_through_a(A, B, k_end, smem, acc);
    } else {
      acc.clear();
      if constexpr (NB == 2) gemm_tile<LOADS, Through::kA, RING>(A, B, 0, k_end, smem, acc);
      else gemm_tile<LOADS>(A, B, 0, k_end, smem, acc);
    }
  }
};

}  // namespace ct
