// Sparse cross-entropy on materialised logits: per-row weighted loss with an online
// log-sum-exp in one pass over HBM, and the analytic logits gradient in one more. The loss
// backend the trainer falls back to when the projection-fused operator is not selected.
//
// Reference: src/kernels/cross_entropy.py:99-190 (_ce_stats_kernel), :254-323 (_ce_bwd_kernel),
// :400-420 (_replicated_loss_and_lse); semantics of the XLA path
// src/kernels/fused_cross_entropy.py:64-106.
#include "ct_error.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ct {

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2eF = 1.4426950408889634f;
constexpr float kLn2F = 0.6931471805599453f;
constexpr float kNegInfinity = -__builtin_inff();

template <class T>
__device__ __forceinline__ float to_f32(T v) { return (float)v; }

// (m, s): running maximum (log2 domain) and sum of exp2(x log2e - m). The exponents are at most 0, so the
// bare instruction serves: what it flushes to 0 is below 2^-126 of the sum.
template <int N>
__device__ __forceinline__ void online_add(float& m, float& s, const float* x) {
  float cm = x[0];
#pragma unroll
  for (int e = 1; e < N; ++e) cm = fmaxf(cm, x[e]);
  cm *= kLog2eF;
  if (cm > m) {
    s *= __builtin_amdgcn_exp2f(m - cm);  // m = -inf: s is 0 and stays 0
    m = cm;
  }
  if (m == kNegInfinity) return;  // only -inf so far
  float t = 0.f;
#pragma unroll
  for (int e = 0; e < N; e += 2) {
    s += __builtin_amdgcn_exp2f(fmaf(x[e], kLog2eF, -m));
    if (e + 1 < N) t += __builtin_amdgcn_exp2f(fmaf(x[e + 1], kLog2eF, -m));
  }
  s += t;
}
__device__ __forceinline__ void online_merge(float& m, float& s, float mo, float so) {
  const float mn = fmaxf(m, mo);
  if (mn == kNegInfinity) return;
  s = s * exp2f(m - mn) + so * exp2f(mo - mn);
  m = mn;
}

// A row as 16-byte chunks: `head` elements in front of the first aligned address (rows of an odd
// vocabulary start anywhere), `chunks` chunks, the rest behind them.
template <class T>
struct RowChunks {
  static constexpr int kPer = 16 / sizeof(T);  // elements per chunk
  int head, chunks;
  __device__ RowChunks(const T* x, int vocab) {
    const int off = (int)(reinterpret_cast<uintptr_t>(x) & 15u) / (int)sizeof(T);
    head = off ? min(vocab, kPer - off) : 0;
    chunks = (vocab - head) / kPer;
  }
};
template <class T>
__device__ __forceinline__ void widen(u32x4 raw, float* v) {
  if constexpr (sizeof(T) == 2) {
    const bf16x8 b = __builtin_bit_cast(bf16x8, raw);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)b[e];
  } else {
    const f32x4 f = __builtin_bit_cast(f32x4, raw);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = f[e];
  }
}

// One workgroup per row. valid = target != ignore_index && weight != 0; invalid rows cost no
// traffic and give loss = lse = 0. A target outside [0, vocab) on a valid row contributes a
// target logit of 0, as the reference's masked lookup does.
// Bound by memory: a thread has kUnroll chunks in flight. Aligned or not, a row is read in whole chunks
// (element by element, as before, the rows of an odd vocabulary ran at 2.2 TB/s).
constexpr int kUnroll = 4;
template <class T, int THREADS>
__global__ __launch_bounds__(THREADS) void sparse_ce_fwd_kernel(const T* logits, const int* targets,
                                                                const float* weights, int vocab,
                                                                int ignore_index,
                                                                float* loss, float* lse) {
  constexpr int kWaves = THREADS / 64;
  __shared__ float wm[kWaves], ws[kWaves];
  const long row = blockIdx.x;
  const int tid = threadIdx.x;
  const int target = targets[row];
  const float weight = weights[row];
  if (target == ignore_index || weight == 0.f) {
    if (tid == 0) {
      loss[row] = 0.f;
      lse[row] = 0.f;
    }
    return;
  }
  const T* x = logits + (size_t)row * vocab;
  float m = kNegInfinity, s = 0.f;
  const RowChunks<T> rc(x, vocab);
  constexpr int kPer = RowChunks<T>::kPer;
  const u32x4* body = reinterpret_cast<const u32x4*>(x + rc.head);
  int c = tid;
  for (; c + (kUnroll - 1) * THREADS < rc.chunks; c += kUnroll * THREADS) {
    u32x4 raw[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) raw[u] = body[c + u * THREADS];
    float v[kUnroll * kPer];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) widen<T>(raw[u], v + u * kPer);
    online_add<kUnroll * kPer>(m, s, v);
  }
  for (; c < rc.chunks; c += THREADS) {
    float v[kPer];
    widen<T>(body[c], v);
    online_add<kPer>(m, s, v);
  }
  // the elements in front of and behind the chunks: fewer than 2 kPer
  const int behind = rc.head + rc.chunks * kPer, loose = rc.head + vocab - behind;
  if (tid < loose) {
    const float v = to_f32(x[tid < rc.head ? tid : behind + tid - rc.head]);
    online_add<1>(m, s, &v);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float mo = __shfl_xor(m, off, 64), so = __shfl_xor(s, off, 64);
    online_merge(m, s, mo, so);
  }
  if ((tid & 63) == 0) {
    wm[tid >> 6] = m;
    ws[tid >> 6] = s;
  }
  __syncthreads();
  if (tid == 0) {
    for (int k = 1; k < kWaves; ++k) online_merge(m, s, wm[k], ws[k]);
    const float row_lse = logf(s) + m * kLn2F;
    const float target_logit = (target >= 0 && target < vocab) ? to_f32(x[target]) : 0.f;
    lse[row] = row_lse;
    loss[row] = weight * (row_lse - target_logit);
  }
}

// grid = (rows, parts of kCeBwdChunks chunks of a row).
// dlogits = w dy (exp(x - lse) - onehot) on valid rows, 0 elsewhere, in the logits dtype.
// STREAM: the tensors are too large to be found in a cache again, so reads and writes bypass it.
constexpr int kCeBwdChunks = 256 * 2 * kUnroll;
template <class T, bool STREAM>
__global__ __launch_bounds__(256) void sparse_ce_bwd_kernel(const T* logits, const float* lse,
                                                            const int* targets, const float* weights,
                                                            const float* dy, int vocab, int ignore_index,
                                                            bool same_alignment, T* dlogits) {
  const long row = blockIdx.x;
  const int tid = threadIdx.x;
  const int target = targets[row];
  const float weight = weights[row];
  const bool valid = target != ignore_index && weight != 0.f;
  const float factor = valid ? weight * dy[row] : 0.f;
  const float lse2 = valid ? lse[row] * kLog2eF : 0.f;
  const T* x = logits + (size_t)row * vocab;
  T* g = dlogits + (size_t)row * vocab;
  constexpr int kPer = RowChunks<T>::kPer;
  auto grad = [&](float v, int index) {
    return factor * (exp2f(fmaf(v, kLog2eF, -lse2)) - (index == target ? 1.f : 0.f));
  };
  // (chunks are aligned in dlogits, where they are written; logits aligned another way are read unaligned)
  const RowChunks<T> rc(g, vocab);
  const int first = blockIdx.y * kCeBwdChunks, last = min(rc.chunks, first + kCeBwdChunks);
  auto load = [&](int c) {
    const T* at = x + rc.head + (size_t)c * kPer;
    u32x4 raw;
    if (!same_alignment) __builtin_memcpy(&raw, at, 16);
    else if (STREAM) raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(at));
    else raw = *reinterpret_cast<const u32x4*>(at);
    return raw;
  };
  auto store = [&](int c, u32x4 out) {
    u32x4* at = reinterpret_cast<u32x4*>(g + rc.head + (size_t)c * kPer);
    if (STREAM) __builtin_nontemporal_store(out, at);
    else *at = out;
  };
  auto gradients = [&](u32x4 raw, int c) {
    float v[kPer];
    widen<T>(raw, v);
    const int i0 = rc.head + c * kPer;
    if constexpr (sizeof(T) == 2) {
      bf16x8 out;
#pragma unroll
      for (int e = 0; e < kPer; ++e) out[e] = (bf16)grad(v[e], i0 + e);
      return __builtin_bit_cast(u32x4, out);
    } else {
      f32x4 out;
#pragma unroll
      for (int e = 0; e < kPer; ++e) out[e] = grad(v[e], i0 + e);
      return __builtin_bit_cast(u32x4, out);
    }
  };
  if (!valid) {
    for (int c = first + tid; c < last; c += 256) store(c, u32x4{0u, 0u, 0u, 0u});
  } else {
    int c = first + tid;
    for (; c + (kUnroll - 1) * 256 < last; c += kUnroll * 256) {
      u32x4 raw[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) raw[u] = load(c + u * 256);
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) store(c + u * 256, gradients(raw[u], c + u * 256));
    }
    for (; c < last; c += 256) store(c, gradients(load(c), c));
  }
  const int behind = rc.head + rc.chunks * kPer, loose = rc.head + vocab - behind;
  if (blockIdx.y == 0 && tid < loose) {
    const int i = tid < rc.head ? tid : behind + tid - rc.head;
    g[i] = (T)(valid ? grad(to_f32(x[i]), i) : 0.f);
  }
}

// Logits larger than the memory-side cache (256 MB) are not found there by the backward.
constexpr size_t kStreamBytes = (size_t)384 << 20;

static int check_ce(const char* fn, const ct_sparse_ce_args* a) {
  CT_REQUIRE(a, "%s: null args", fn);
  CT_REQUIRE(a->logits && a->targets && a->weights, "%s: null pointer", fn);
  CT_REQUIRE(a->rows > 0 && a->vocab > 0, "%s: logits must have at least one row and one column", fn);
  CT_REQUIRE(a->logits_dtype == CT_DTYPE_BF16 || a->logits_dtype == CT_DTYPE_F32,
             "%s: logits must be bfloat16 or float32", fn);
  CT_REQUIRE(a->rows <= 0x7fffffffLL, "%s: at most 2^31 - 1 rows", fn);
  CT_REQUIRE(reinterpret_cast<uintptr_t>(a->logits) % (a->logits_dtype == CT_DTYPE_BF16 ? 2 : 4) == 0,
             "%s: logits must be aligned to their element size", fn);
  return CT_OK;
}

}  // namespace ct

using namespace ct;

extern "C" int32_t ct_sparse_ce_fwd(void* stream_, const ct_sparse_ce_args* a, float* loss, float* lse) {
  int rc = check_ce("ct_sparse_ce_fwd", a);
  if (rc) return rc;
  CT_REQUIRE(loss && lse, "ct_sparse_ce_fwd: null output");
  hipStream_t stream = (hipStream_t)stream_;
  LaunchScope scope("sparse_ce_fwd_kernel", stream);
  // few rows leave compute units without a workgroup: then a row gets four times the threads
  const bool wide = a->rows <= 512 && a->vocab >= 8192;
  const auto launch = [&](auto kernel, auto* logits) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)a->rows), dim3(wide ? 1024 : 256), 0, stream, logits, a->targets, a->weights,
                       a->vocab, a->ignore_index, loss, lse);
  };
  if (a->logits_dtype == CT_DTYPE_BF16)
    launch(wide ? sparse_ce_fwd_kernel<bf16, 1024> : sparse_ce_fwd_kernel<bf16, 256>, static_cast<const bf16*>(a->logits));
  else
    launch(wide ? sparse_ce_fwd_kernel<float, 1024> : sparse_ce_fwd_kernel<float, 256>, static_cast<const float*>(a->logits));
  return scope.done();
}

extern "C" int32_t ct_sparse_ce_bwd(void* stream_, const ct_sparse_ce_args* a, const float* lse,
                                    const float* dy, void* dlogits) {
  int rc = check_ce("ct_sparse_ce_bwd", a);
  if (rc) return rc;
  CT_REQUIRE(lse && dy && dlogits, "ct_sparse_ce_bwd: null pointer");
  hipStream_t stream = (hipStream_t)stream_;
  const size_t elem = a->logits_dtype == CT_DTYPE_BF16 ? 2 : 4;
  CT_REQUIRE(reinterpret_cast<uintptr_t>(dlogits) % elem == 0, "ct_sparse_ce_bwd: dlogits must be aligned to its element size");
  const bool same = ((reinterpret_cast<uintptr_t>(a->logits) ^ reinterpret_cast<uintptr_t>(dlogits)) & 15u) == 0;
  const bool stream_through = (size_t)a->rows * a->vocab * elem > kStreamBytes;
  const int chunks = (int)(a->vocab * elem / 16);
  const dim3 grid((unsigned)a->rows, (unsigned)(chunks > kCeBwdChunks ? (chunks + kCeBwdChunks - 1) / kCeBwdChunks : 1));
  LaunchScope scope("sparse_ce_bwd_kernel", stream);
  const auto launch = [&](auto kernel, auto* out) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, static_cast<decltype(out)>(const_cast<void*>(a->logits)), lse, a->targets,
                       a->weights, dy, a->vocab, a->ignore_index, same, out);
  };
  if (a->logits_dtype == CT_DTYPE_BF16)
    launch(stream_through ? sparse_ce_bwd_kernel<bf16, true> : sparse_ce_bwd_kernel<bf16, false>, static_cast<bf16*>(dlogits));
  else
    launch(stream_through ? sparse_ce_bwd_kernel<float, true> : sparse_ce_bwd_kernel<float, false>, static_cast<float*>(dlogits));
  return scope.done();
}
