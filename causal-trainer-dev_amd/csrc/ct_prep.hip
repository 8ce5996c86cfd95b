// Device-side preparation steps that sit directly in front of the two hot paths and define
// their ignored-token sets: segment id canonicalisation and shifted targets / loss weights.
// Integer work, bit-exact against the reference (src/modeling/rotary.py:13-50,
// src/training/losses.py:21-85).
#include "ct_error.h"
#include "ct_lanes.hip.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ct {

// One workgroup per batch row, kScanPer consecutive positions per thread and pass. A run starts at a
// valid position (mask != 0) whose predecessor is invalid or carries a different label (position 0
// compares its label with itself, as the reference does).
// POSITIONS = false: out[s] = number of run starts in [0, s] where s is valid, else 0;
// POSITIONS = true:  out[s] = s - the latest run start where s is valid, else 0.
// The time is that of the passes' chains (load, scan in the wavefront, exchange, store): 4096 positions
// take one pass. Rows at 16-byte addresses are moved in quads (ALIGNED), scans and exchanges are lane moves of the vector
// ALU, where a shuffle through LDS has ten times the latency: [4, 4096] 5.5 -> 4.0 us.
constexpr int kScanPer = 4;
template <bool POSITIONS, bool ALIGNED>
__global__ __launch_bounds__(1024) void segment_scan_kernel(const int* mask, const int* labels, int S, int* out) {
  __shared__ int wave_total[2][16];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwaves = blockDim.x >> 6;
  const int* mrow = mask + (size_t)b * S;
  const int* lrow = labels ? labels + (size_t)b * S : nullptr;
  int* orow = out + (size_t)b * S;
  int carry = 0;  // of the passes before: run starts so far / the latest start
  for (int base = 0, pass = 0; base < S; base += blockDim.x * kScanPer, ++pass) {
    const int s0 = base + tid * kScanPer;
    int m[kScanPer + 1], l[kScanPer + 1];
    if constexpr (ALIGNED) {  // (S is a multiple of 4: all of a thread's positions or none)
      const bool in = s0 < S, before = lane == 0 && s0 > 0 && in;
      const int4 zero = {0, 0, 0, 0};
      const int4 mv = in ? *reinterpret_cast<const int4*>(mrow + s0) : zero;
      const int4 lv = lrow && in ? *reinterpret_cast<const int4*>(lrow + s0) : zero;
      const int m_before = before ? mrow[s0 - 1] : 0, l_before = lrow && before ? lrow[s0 - 1] : 0;
      m[1] = mv.x, m[2] = mv.y, m[3] = mv.z, m[4] = mv.w;
      l[1] = lv.x, l[2] = lv.y, l[3] = lv.z, l[4] = lv.w;
      m[0] = lane_below(mv.w, m_before);
      l[0] = lane_below(lv.w, l_before);
    } else {
#pragma unroll
      for (int k = 0; k <= kScanPer; ++k) {
        const int s = s0 + k - 1;
        const bool in = s >= 0 && s < S;
        m[k] = in ? mrow[s] : 0;
        l[k] = lrow && in ? lrow[s] : 0;
      }
    }
    int run[kScanPer], mine = 0;
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) {
      const bool start = m[k + 1] != 0 && (m[k] == 0 || l[k + 1] != l[k]);
      mine = POSITIONS ? max(mine, start ? s0 + k : 0) : mine + start;
      run[k] = mine;
    }
    const int incl = wave_scan<POSITIONS>(mine);
    int* total = wave_total[pass & 1];  // (two of them: one barrier per pass)
    if (lane == 63) total[wave] = incl;
    __syncthreads();
    const int totals = wave_scan<POSITIONS>(lane < nwaves ? total[lane] : 0);
    int before = wave ? lane_value(totals, wave - 1) : 0;
    before = POSITIONS ? max(before, carry) : before + carry;
    const int all = lane_value(totals, nwaves - 1);
    carry = POSITIONS ? max(carry, all) : carry + all;
    const int left = lane_below(incl, 0);
    before = POSITIONS ? max(before, left) : before + left;
    int value[kScanPer];
#pragma unroll
    for (int k = 0; k < kScanPer; ++k)
      value[k] = m[k + 1] == 0 ? 0 : POSITIONS ? s0 + k - max(before, run[k]) : before + run[k];
    if constexpr (ALIGNED) {
      if (s0 < S) *reinterpret_cast<int4*>(orow + s0) = int4{value[0], value[1], value[2], value[3]};
    } else {
#pragma unroll
      for (int k = 0; k < kScanPer; ++k)
        if (s0 + k < S) orow[s0 + k] = value[k];
    }
  }
}

// targets[b, s] = labels[b, s + 1] where the weight is positive, else 0;
// weights[b, s] = valid edge * assistant[s + 1] * loss_mask[s + 1]  (f32 products in that order).
// Two neighbours lie in the same canonical run iff both are valid (mask == 1 here, not != 0:
// src/training/losses.py:52) and carry the same label, so no run ids are needed.
__global__ __launch_bounds__(256) void shifted_targets_kernel(
    const int* input_ids, const int* labels, const int* mask, const int* segments,
    const int* assistant, const float* loss_mask, int ignore_index, int B, int S, int* targets,
    float* weights) {
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  const long total = (long)B * (S - 1);
  if (gid >= total) return;
  const int b = (int)(gid / (S - 1)), s = (int)(gid % (S - 1));
  const size_t here = (size_t)b * S + s, next = here + 1;
  const int* lab = labels ? labels : input_ids;
  const int target = lab[next];
  bool valid = target != ignore_index;
  if (mask) valid = valid && mask[here] == 1 && mask[next] == 1;
  if (segments) valid = valid && segments[here] == segments[next];
  float w = valid ? 1.f : 0.f;
  if (assistant) w *= (assistant[next] != 0) ? 1.f : 0.f;
  if (loss_mask) w *= loss_mask[next];
  weights[gid] = w;
  targets[gid] = w > 0.f ? target : 0;
}

static int check_dims(const char* fn, int batch, int seq) {
  CT_REQUIRE(batch > 0 && seq > 0, "%s: batch and sequence must be positive, got [%d, %d]", fn,
             batch, seq);
  return CT_OK;
}

template <bool POSITIONS>
static int launch_segment_scan(hipStream_t stream, const char* name, const int* mask, const int* labels, int batch, int seq,
                               int* out) {
  const int needed = (seq + kScanPer - 1) / kScanPer, threads = needed >= 1024 ? 1024 : ((needed + 63) / 64) * 64;
  const bool aligned = seq % 4 == 0 && ((reinterpret_cast<uintptr_t>(mask) | reinterpret_cast<uintptr_t>(labels) |
                                         reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
  LaunchScope scope(name, stream);
  hipLaunchKernelGGL((aligned ? segment_scan_kernel<POSITIONS, true> : segment_scan_kernel<POSITIONS, false>), dim3(batch), dim3(threads), 0, stream, mask, labels, seq, out);
  return scope.done();
}

// Transposed copy of 16-bit elements: dst [cols][ld], of whose rows the first `rows` elements are src [rows][cols]^T and
// the others zero. Bound by memory. A workgroup
// takes a 64 x 64 tile, so both sides move whole 128-byte lines; a thread loads 8 columns of two rows and
// stores 8 rows of two columns (memcpy: rows of an odd length start at any multiple of 2 bytes, which an
// ordinary access may). LDS rows are 66 elements: the 8-element columns that a wavefront collects lie
// 8 * 33 words apart per lane group and hit all banks. [76395, 1536]: 119 us (4.0 TB/s; a strided copy of the
// transposed view 2264), [32000, 4096]: 116 us (4.5 TB/s; 1859).
constexpr int kTransposeTile = 64, kTransposePitch = kTransposeTile + 2;
__global__ __launch_bounds__(256) void transpose16_kernel(const unsigned short* src, int rows, int cols, unsigned short* dst, int ld) {
  __shared__ unsigned short tile[kTransposeTile * kTransposePitch];
  const unsigned col_tiles = ((unsigned)cols + kTransposeTile - 1) / kTransposeTile;
  const int r0 = (int)(blockIdx.x / col_tiles) * kTransposeTile, c0 = (int)(blockIdx.x % col_tiles) * kTransposeTile;
  const int line = threadIdx.x >> 3, chunk = (threadIdx.x & 7) * 8;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int r = line + 32 * pass, left = r0 + r < rows ? cols - (c0 + chunk) : 0;
    const unsigned short* from = src + (size_t)(r0 + r) * cols + c0 + chunk;
    unsigned short v[8] = {};
    if (left >= 8) {
      __builtin_memcpy(v, from, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < left) v[e] = from[e];
    }
#pragma unroll
    for (int e = 0; e < 8; e += 2)
      *reinterpret_cast<unsigned*>(&tile[r * kTransposePitch + chunk + e]) = v[e] | (unsigned)v[e + 1] << 16;
  }
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int c = line + 32 * pass, left = c0 + c < cols ? ld - (r0 + chunk) : 0;
    unsigned short* to = dst + (size_t)(c0 + c) * ld + r0 + chunk;
    unsigned short v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = tile[(chunk + e) * kTransposePitch + c];
    if (left >= 8) {
      __builtin_memcpy(to, v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < left) to[e] = v[e];
    }
  }
}

}  // namespace ct

using namespace ct;

extern "C" int32_t ct_canonicalize_segment_ids(void* stream, const int32_t* attention_mask,
                                               const int32_t* segment_ids, int32_t batch,
                                               int32_t seq, int32_t* canonical_ids) {
  CT_REQUIRE(attention_mask && canonical_ids, "ct_canonicalize_segment_ids: null pointer");
  int rc = check_dims("ct_canonicalize_segment_ids", batch, seq);
  if (rc) return rc;
  return launch_segment_scan<false>((hipStream_t)stream, "canonicalize_kernel", attention_mask, segment_ids, batch, seq,
                                    canonical_ids);
}

extern "C" int32_t ct_segment_positions(void* stream, const int32_t* attention_mask, const int32_t* segment_ids,
                                        int32_t batch, int32_t seq, int32_t* position_ids) {
  CT_REQUIRE(attention_mask && position_ids, "ct_segment_positions: null pointer");
  int rc = check_dims("ct_segment_positions", batch, seq);
  if (rc) return rc;
  return launch_segment_scan<true>((hipStream_t)stream, "segment_positions_kernel", attention_mask, segment_ids, batch, seq,
                                   position_ids);
}

extern "C" size_t ct_shifted_targets_scratch_bytes(int32_t batch, int32_t seq) {
  (void)batch;
  (void)seq;
  return 0;  // (the kernel compares neighbours and needs none)
}

extern "C" int32_t ct_shifted_targets_and_weights(void* stream_, const ct_shifted_targets_args* a) {
  CT_REQUIRE(a, "ct_shifted_targets_and_weights: null args");
  CT_REQUIRE(a->input_ids && a->targets && a->weights, "ct_shifted_targets_and_weights: null pointer");
  int rc = check_dims("ct_shifted_targets_and_weights", a->batch, a->seq);
  if (rc) return rc;
  CT_REQUIRE(a->seq >= 2, "ct_shifted_targets_and_weights: sequence length %d leaves no prediction edge",
             a->seq);
  hipStream_t stream = (hipStream_t)stream_;
  const long total = (long)a->batch * (a->seq - 1);
  LaunchScope scope2("shifted_targets_kernel", stream);
  hipLaunchKernelGGL(shifted_targets_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream,
                     a->input_ids, a->labels, a->attention_mask, a->segment_ids, a->assistant_mask,
                     a->loss_mask, a->ignore_index, a->batch, a->seq, a->targets, a->weights);
  return scope2.done();
}

extern "C" int32_t ct_transpose16(void* stream, const uint16_t* src, int32_t rows, int32_t cols, uint16_t* dst) {
  return ct_transpose16_padded(stream, src, rows, cols, dst, rows);
}
extern "C" int32_t ct_transpose16_padded(void* stream_, const uint16_t* src, int32_t rows, int32_t cols, uint16_t* dst,
                                         int32_t ld) {
  CT_REQUIRE(src && dst, "ct_transpose16: null pointer");
  CT_REQUIRE(rows > 0 && cols > 0, "ct_transpose16: dimensions must be positive");
  CT_REQUIRE(ld >= rows, "ct_transpose16: rows of %d elements do not fit in %d", rows, ld);
  const long tiles = (long)(((unsigned)ld + kTransposeTile - 1) / kTransposeTile) * (((unsigned)cols + kTransposeTile - 1) / kTransposeTile);
  CT_REQUIRE(tiles <= 0x7fffffff, "ct_transpose16: [%d, %d] has more tiles than a launch takes", rows, cols);
  LaunchScope scope("transpose16_kernel", (hipStream_t)stream_);
  hipLaunchKernelGGL(transpose16_kernel, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream_, src, rows, cols, dst, ld);
  return scope.done();
}
