// 256 x 256 workgroup-tile bf16 GEMM core for gfx950, used by the cut
// cross-entropy kernels.
//
// 4 wavefronts in a 2 x 2 arrangement, 128 x 128 outputs per wavefront held
// as 4 x 4 mfma32 accumulator blocks (256 f32 registers per lane). The
// contraction runs in steps of BK = 32.
//
// An operand comes in one of two memory layouts:
//   KcLoader  "k-contiguous": matrix rows are the M (or N) index, the
//             contraction index is contiguous. LDS tile [256][BK], MFMA
//             fragments read with ds_read_b128.
//   McLoader  "m-contiguous": matrix rows are the contraction index, the M
//             (or N) index is contiguous. LDS tile [BK][256], fragments read
//             with transposed LDS reads.
// The rows of a k-contiguous operand can be addressed through an index list (gather).
//
// Two main loops share the loaders; a kernel is compiled for one of them (GUARDED), because both in
// one kernel cost it registers, spills and instruction cache:
//   pipelined  operands 16-byte aligned, contraction a multiple of 128: tiles are copied global ->
//              LDS asynchronously, three steps ahead, into a ring of 4 LDS stages; MFMA fragments
//              are double buffered in registers so that LDS reads of the next half step overlap
//              the 16 MFMAs of the current one; one barrier per step (gen_gemm_asm.py). Rows or
//              columns of a tile past the end of the matrix are copies of valid ones.
//   guarded    unaligned operands: element-wise guarded loads that zero fill, staged through
//              registers, 2 LDS stages.
#pragma once

#include "ct_common.hip.h"
#include "ct_gemm_asm.inc"

namespace ct {

constexpr int kGemmTile = 256;
constexpr int kGemmBK = 32;

CT_DEVICE u32x4 load_chunk_guarded(const bf16* p, int count) {
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = e < count ? p[e] : (bf16)0.f;
  return as_u32x4(v);
}

struct GemmSmem {
  static constexpr int kTileBytes = kGemmTile * kGemmBK * 2;  // 16 KB
  static constexpr int kStageBytes = 2 * kTileBytes;          // A tile then B tile
  static constexpr int kStages = 4;
  static constexpr size_t kBytes = (size_t)kStages * kStageBytes;  // 128 KB
};

// In both loaders thread t owns the 16-byte LDS slots t + 256 n of the tile
// (n < 4): slot P holds physical chunk P % CPR of row P / CPR, i.e. logical
// chunk (P % CPR) ^ swizzle(row); voff[n] is the byte offset of that chunk
// from `base` at k = 0 (32 bits: the host checks sizes and strides against it).
struct KcLoader {
  static constexpr int CPR = kGemmBK / 8;  // 4
  static constexpr int NCH = 4;
  const char* base;    // uniform
  unsigned voff[NCH];
  u32x4 regs[NCH];
  int chunk, k_valid;

  // rows m0 .. m0+255 of `base_` (leading dimension ld elements), optionally
  // gathered through row_index. Rows >= rows_valid are copies of the first row (callers discard
  // what they get from them); the guarded loop reads k >= k_valid as zero.
  // With interleave_rows, tile row 128 w + 32 nb + j holds matrix row m0 + 128 w + 4 j + nb:
  // in the accumulator layout lane j of a wavefront then owns 4 consecutive matrix rows (its
  // column blocks nb = 0..3), which an epilogue can store with one 8- or 16-byte access.
  CT_DEVICE void init(const bf16* base_, long ld, const int* row_index, int m0, int rows_valid,
                      int k_valid_, bool interleave_rows = false) {
    const int t = threadIdx.x;
    k_valid = k_valid_;
    const bool gathered = row_index != nullptr;
    base = reinterpret_cast<const char*>(gathered ? base_ : base_ + (size_t)m0 * ld);
    const int r0 = t / CPR;
    chunk = (t % CPR) ^ swizzle<CPR>(r0);  // rows r0 + 64 n share the swizzle
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      const int tile_row = r0 + 64 * n;
      const int r = interleave_rows ? ((tile_row & 128) | ((tile_row & 31) << 2) | ((tile_row >> 5) & 3))
                                    : tile_row;
      const bool ok = m0 + r < rows_valid;
      const long src = gathered ? row_index[ok ? m0 + r : 0] : (ok ? r : 0);
      voff[n] = (unsigned)((src * ld + chunk * 8) * 2);
    }
  }
  // copies N0 .. N1-1 of the thread's NCH 16-byte slots
  template <int N0 = 0, int N1 = NCH>
  CT_DEVICE void dma(int k0, lds_addr tile) const {
    const int wave = uniform(threadIdx.x >> 6);
    const char* p = base + (size_t)k0 * 2;
#pragma unroll
    for (int n = N0; n < N1; ++n) dma16_s(p, voff[n], tile + (n * 256 + wave * 64) * 16);
  }
  CT_DEVICE void fetch(int k0) {
    const int k = k0 + chunk * 8;
    const int count = min(max(k_valid - k, 0), 8);
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      regs[n] = count ? load_chunk_guarded(reinterpret_cast<const bf16*>(
                                                       base + (size_t)k0 * 2 + voff[n]),
                                                   count)
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

struct McLoader {
  static constexpr int CPR = kGemmTile / 8;  // 32
  static constexpr int NCH = 4;
  const char* base;  // uniform: column m0 of row 0
  long ld;
  unsigned voff[NCH];
  u32x4 regs[NCH];
  int col[2];  // first column of the chunk fetched in even / odd passes
  int cols_left, k_valid;

  // columns m0 .. m0+255 of `base_`. The guarded loop reads columns >= cols_valid and rows >= k_valid
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
      const int r = t / CPR + 8 * n;
      int c = ((t % CPR) ^ swizzle<CPR>(r)) * 8;
      col[n & 1] = c;
      if (c >= cols_left) c = 0;
      voff[n] = (unsigned)(((long)r * ld + c) * 2);
    }
  }
  // copies N0 .. N1-1 of the thread's NCH 16-byte slots (N0 even, N1 = N0 + 2 or NCH)
  template <int N0 = 0, int N1 = NCH>
  CT_DEVICE void dma(int k0, lds_addr tile) const {
    const int wave = uniform(threadIdx.x >> 6);
    const char* p = base + (size_t)k0 * ld * 2;
#pragma unroll
    for (int n = N0; n < N1; ++n) dma16_s(p, voff[n], tile + (n * 256 + wave * 64) * 16);
  }
  CT_DEVICE void fetch(int k0) {
    const int r0 = (int)threadIdx.x / CPR;
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      const int k = k0 + r0 + 8 * n;
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

struct GemmAcc {
  f32x16 c[4][4];
  CT_DEVICE void clear() {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) c[a][b] = zero16();
  }
  // Wait states between the compiler's last MFMA and value(), whose read it does not see.
  CT_DEVICE void settle() {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) asm volatile("" : "+a"(c[a][b]));
    asm volatile("s_nop 15\n\ts_nop 7");
  }
  // An element, read where the call stands. (An epilogue's branches otherwise have the reads and what
  // is computed from them moved in front of the branch, where 256 of them do not fit and spill.)
  CT_DEVICE float value(int i, int nb, int r) const {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(c[i][nb][r]));
    return v;
  }
  CT_DEVICE f32x4 quad(int i, int r) const { return f32x4{value(i, 0, r), value(i, 1, r), value(i, 2, r), value(i, 3, r)}; }
};

struct GemmFrags {
  bf16x8 a[4], b[4];
};

template <class ALoader, class BLoader>
CT_DEVICE void load_frags(GemmFrags& f, int stage_off, const typename ALoader::FragOffsets& afo,
                          const typename BLoader::FragOffsets& bfo, int ks, int wm, int wn) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f.a[i] = ALoader::frag(stage_off, afo, ks, wm, i);
    f.b[i] = BLoader::frag(stage_off + GemmSmem::kTileBytes, bfo, ks, wn, i);
  }
}

CT_DEVICE void mfma_block(const GemmFrags& f, GemmAcc& acc) {
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
// m-contiguous A, a k-contiguous B and a step count that is a positive multiple of 4. Entered with the copies of steps 0..2 issued and step 0 landed for every
// wavefront; returns with nothing in flight and the LDS tiles free.
CT_DEVICE unsigned long long uniform64(const void* p) {
  const unsigned long long b = (unsigned long long)(uintptr_t)p;
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
  return ((unsigned long long)hi << 32) | (unsigned long long)lo;
}
CT_DEVICE void gemm_loop_scheduled(const McLoader& A, const KcLoader& B, int k_begin, int steps,
                                   lds_addr smem, const McLoader::FragOffsets& afo,
                                   const KcLoader::FragOffsets& bfo, int wm, int wn, GemmAcc& acc) {
  const int wave = uniform(threadIdx.x >> 6);
  // sources of the copies of step 3
  const unsigned long long src_a =
      uniform64(A.base + (size_t)(k_begin + 3 * kGemmBK) * (size_t)A.ld * 2);
  const unsigned long long src_b = uniform64(B.base + (size_t)(k_begin + 3 * kGemmBK) * 2);
  const unsigned stride_a = (unsigned)uniform((int)(kGemmBK * A.ld * 2));
  const unsigned steps_u = (unsigned)uniform(steps);
  const unsigned lds_wave = (unsigned)uniform((int)(uintptr_t)(smem + wave * 1024));
  const int a_off = (wm / 128) * 256;
  const int b_off = GemmSmem::kTileBytes + (wn / 32) * KcLoader::FragOffsets::kRowBlockBytes;
  asm volatile(CT_GEMM_LOOP
               : "+a"(acc.c[0][0]), "+a"(acc.c[0][1]), "+a"(acc.c[0][2]), "+a"(acc.c[0][3]),
                 "+a"(acc.c[1][0]), "+a"(acc.c[1][1]), "+a"(acc.c[1][2]), "+a"(acc.c[1][3]),
                 "+a"(acc.c[2][0]), "+a"(acc.c[2][1]), "+a"(acc.c[2][2]), "+a"(acc.c[2][3]),
                 "+a"(acc.c[3][0]), "+a"(acc.c[3][1]), "+a"(acc.c[3][2]), "+a"(acc.c[3][3])
               : "s"(src_a), "s"(src_b), "s"(stride_a), "s"(steps_u), "s"(lds_wave),
                 "v"(afo.ptr[0][0] + a_off), "v"(afo.ptr[0][1] + a_off), "v"(afo.ptr[0][2] + a_off),
                 "v"(afo.ptr[0][3] + a_off), "v"(afo.ptr[1][0] + a_off), "v"(afo.ptr[1][1] + a_off),
                 "v"(afo.ptr[1][2] + a_off), "v"(afo.ptr[1][3] + a_off), "v"(bfo.ptr[0] + b_off),
                 "v"(bfo.ptr[1] + b_off), "v"(A.voff[0]), "v"(A.voff[1]), "v"(A.voff[2]),
                 "v"(A.voff[3]), "v"(B.voff[0]), "v"(B.voff[1]), "v"(B.voff[2]), "v"(B.voff[3])
               : "memory", "m0", "scc", CT_GEMM_LOOP_CLOBBERS);
}

// acc += A[m-tile, k_begin:k_end] * B[n-tile, k_begin:k_end]^T (k_end - k_begin a multiple of 128
// unless GUARDED). Must be called by all 256 threads; ends with the LDS tiles free for reuse.
template <bool GUARDED>
CT_DEVICE void gemm_tile(McLoader& A, KcLoader& B, int k_begin, int k_end, lds_addr smem, GemmAcc& acc) {
  constexpr int BK = kGemmBK, kTile = GemmSmem::kTileBytes, kStage = GemmSmem::kStageBytes;
  const int w = threadIdx.x >> 6;
  const int wm = (w >> 1) * 128, wn = (w & 1) * 128;
  if (k_begin >= k_end) return;
  const McLoader::FragOffsets afo(smem);
  const KcLoader::FragOffsets bfo(smem);
  if constexpr (!GUARDED) {
    dma_wait_all();  // nothing of ours may still be in flight when counting copies below
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      A.dma(k_begin + i * BK, smem + i * kStage);
      B.dma(k_begin + i * BK, smem + i * kStage + kTile);
    }
    static_assert(McLoader::NCH + KcLoader::NCH == 8, "the wait leaves the copies of two steps in flight");
    wait_vmcnt16();
    workgroup_barrier();
    gemm_loop_scheduled(A, B, k_begin, (k_end - k_begin) / BK, smem, afo, bfo, wm, wn, acc);
  } else {
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
        load_frags<McLoader, KcLoader>(f, cur, afo, bfo, ks, wm, wn);
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

}  // namespace ct
