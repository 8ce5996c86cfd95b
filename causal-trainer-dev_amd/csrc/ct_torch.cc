// The torch side of the operators in native code: argument checks of the usual case, allocation of
// outputs and scratch, the calls into the C ABI, and the autograd nodes. Built by build.py into
// _native.so beside libct_hotpath.so, which it links; host code only.
//
// Why: at the small end a pass is host time. An operator written as a Python autograd function with
// ctypes structures cost 60-90 us per call and direction (measured: attention at [2, 1024, 8, 64] 171 us a
// pass for 75 us of kernels, RMS norm and rotary on 260 tokens 207 us for 35); here it is 5-10.
//
// Every operator function returns None when its arguments are not the plain case it takes (another
// dtype, device, layout or shape): the Python wrapper then runs the full validation, which raises
// or normalises, and calls again.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/extension.h>

#include <cmath>
#include <exception>
#include <mutex>
#include <optional>
#include <tuple>

#include "../../include/ct_hotpath.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
typedef std::optional<Tensor> MaybeTensor;

struct StatusError : std::exception {
  int status;
  std::string message, text;
  explicit StatusError(int s) : status(s), message(ct_last_error()) {
    text = "[ct_status " + std::to_string(s) + "] " + message;
  }
  const char* what() const noexcept override { return text.c_str(); }
};
inline void check(int status) {
  if (status != CT_OK) throw StatusError(status);
}

py::handle error_class;  // CtError of _lib.py, kept for the life of the process
// Makes `e` the current Python error (the caller holds the GIL).
void set_python_error(const StatusError& e) {
  if (!error_class) return PyErr_SetString(PyExc_RuntimeError, e.what());
  py::object error = error_class(e.status, e.message);
  PyErr_SetObject(error_class.ptr(), error.ptr());
}

// A node whose library errors reach the caller of the backward as CtError: autograd hands on Python
// errors as they are and any other exception as a plain RuntimeError.
struct OperatorNode : Node {
  virtual variable_list differentiate(variable_list&& grads) = 0;
  variable_list apply(variable_list&& grads) final {
    try {
      return differentiate(std::move(grads));
    } catch (const StatusError& e) {
      py::gil_scoped_acquire gil;
      set_python_error(e);
      python_error raised;
      raised.persist();  // (this thread's Python state may end with the GIL's release)
      throw raised;
    }
  }
};

inline void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Whether the current stream is being captured into a graph.
inline bool capturing() {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream().stream(), &status) == hipSuccess)
    return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();  // (the default stream while another one is captured)
  return true;
}

template <class T>
inline T* ptr(const Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}
template <class T>
inline T* ptr(const MaybeTensor& t) {
  return t && t->defined() ? static_cast<T*>(t->data_ptr()) : nullptr;
}
inline uint16_t* bits(const Tensor& t) { return ptr<uint16_t>(t); }

inline bool plain(const Tensor& t, at::ScalarType dtype, int64_t dim) {
  return t.defined() && t.is_cuda() && t.scalar_type() == dtype && t.dim() == dim && t.is_contiguous() &&
         t.layout() == at::kStrided && !t.is_neg() && !t.is_conj() &&
         !t._fw_grad(0).defined();  // (the operators have no forward-mode derivative: refused, not dropped)
}
inline Tensor scratch(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte).requires_grad(false));
}
inline Tensor floats(at::IntArrayRef shape, const Tensor& like) {
  return at::empty(shape, like.options().dtype(at::kFloat).requires_grad(false));
}
inline Tensor ints(at::IntArrayRef shape, const Tensor& like) {
  return at::empty(shape, like.options().dtype(at::kInt).requires_grad(false));
}
inline Tensor fresh(const Tensor& like) { return at::empty(like.sizes(), like.options().requires_grad(false)); }
// The incoming gradient of an output, as the kernels take it (zeros where autograd has none).
inline Tensor gradient(const Tensor& grad, at::IntArrayRef shape, at::ScalarType dtype, const Tensor& like) {
  if (!grad.defined()) return at::zeros(shape, like.options().dtype(dtype).requires_grad(false));
  return grad.to(dtype).contiguous();
}

// Attaches `node` to the graph if any input needs a gradient.
template <class N>
std::shared_ptr<N> graph_node(std::initializer_list<Tensor> inputs) {
  std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
  torch::autograd::edge_list edges;
  edges.reserve(inputs.size());
  for (const Tensor& t : inputs) edges.push_back(torch::autograd::impl::gradient_edge(t));
  node->set_next_edges(std::move(edges));
  return node;
}
inline bool needs_graph(std::initializer_list<Tensor> inputs) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : inputs)
    if (t.defined() && t.requires_grad()) return true;
  return false;
}

// ---------------------------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------------------------

// Scratch of the attention backward kept from call to call (BackwardWorkspace in Python), and what the
// dK/dV work list in it was built from. The metadata tensor is held, not remembered by its address: an
// address goes to the next batch's metadata as soon as the last one's are dropped. Writes to it in place
// show in its version counter (inference tensors have none: their list is built on every call).
struct KeptWorkspace {
  std::mutex mutex;  // held while a call chooses, launches and records
  Tensor buffer;
  Tensor listed;  // undefined: no list
  std::tuple<uint32_t, std::vector<int64_t>, int, size_t, float> listed_for;
};

struct AttnShape {
  int32_t batch, seq, q_heads, kv_heads, head_dim;
};
AttnShape attn_shape(const Tensor& q, const Tensor& k) {
  return {(int32_t)q.size(0), (int32_t)q.size(1), (int32_t)q.size(2), (int32_t)k.size(2), (int32_t)q.size(3)};
}

std::tuple<Tensor, Tensor> attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& segments,
                                             const MaybeTensor& ends, const Tensor& bounds, double scale) {
  const c10::DeviceGuard guard(q.device());
  const AttnShape s = attn_shape(q, k);
  Tensor out = fresh(q), lse = floats({s.batch, s.seq, s.q_heads}, q);
  ct_attn_fwd_args a = {};
  a.q = bits(q);
  a.k = bits(k);
  a.v = bits(v);
  a.segment_ids = ptr<int32_t>(segments);
  a.attention_end = ptr<int32_t>(ends);
  a.tile_meta = ptr<int32_t>(bounds);
  a.out = bits(out);
  a.lse = ptr<float>(lse);
  a.batch = s.batch;
  a.seq = s.seq;
  a.q_heads = s.q_heads;
  a.kv_heads = s.kv_heads;
  a.head_dim = s.head_dim;
  a.scale = (float)scale;
  check(ct_attn_fwd(current_stream(), &a));
  return {out, lse};
}

// Left to itself (neither form nor size given) the backward offers the library the larger workspace of
// the stored-dS form for rows of up to CT_ATTN_FROM_DS_UP_TO_SEQ positions, if that is at most 4 GiB: the library
// then takes that form.
constexpr size_t kFromDsWorkspaceCap = (size_t)4 << 30;

// variant: CT_ATTN_BWD_* values; workspace_bytes < 0: what the library asks for the form. A stored-dS form that
// the caller did not pin (no form in `variant`, or form_is_free) gives way to the recomputing one, which needs
// little scratch, where the device has no room for its blocks.
std::tuple<Tensor, Tensor, Tensor, Tensor> attention_backward(const Tensor& q, const Tensor& k, const Tensor& v,
                                                              const Tensor& segments, const MaybeTensor& ends,
                                                              const Tensor& bounds, const Tensor& out, const Tensor& lse,
                                                              const Tensor& dout, double scale, int variant,
                                                              int64_t workspace_bytes, KeptWorkspace* kept,
                                                              bool form_is_free) {
  const c10::DeviceGuard guard(q.device());
  const AttnShape s = attn_shape(q, k);
  const int form = variant & 0xf0;
  const size_t least = ct_attn_bwd_workspace_bytes(s.batch, s.seq, s.q_heads, s.kv_heads, s.head_dim);
  size_t bytes;
  if (workspace_bytes >= 0) {
    bytes = (size_t)workspace_bytes;
  } else {
    const size_t stored = form == CT_ATTN_BWD_DQ_RECOMPUTE || (form == 0 && s.seq > CT_ATTN_FROM_DS_UP_TO_SEQ)
                              ? 0
                              : ct_attn_bwd_workspace_bytes_from_ds(s.batch, s.seq, s.q_heads, s.kv_heads, s.head_dim,
                                                                    ends && ends->defined());
    if (form == CT_ATTN_BWD_DQ_FROM_DS) {
      if (stored == 0)
        throw py::value_error("dq_form='from_ds' is not available for this shape (dS blocks of one KV head "
                              "exceed 64 GiB)");
      bytes = stored;
    } else {
      bytes = stored > 0 && stored <= kFromDsWorkspaceCap ? stored : least;
    }
  }
  Tensor dq = fresh(q), dk = fresh(k), dv = fresh(v), delta = fresh(lse), workspace;
  // (A graph keeps the addresses it was captured with and runs its kernels out of order with later calls:
  // it gets scratch of its own, from its own pool, and builds its own lists.)
  if (kept && capturing()) kept = nullptr;
  const std::unique_lock<std::mutex> lock = kept ? std::unique_lock<std::mutex>(kept->mutex) : std::unique_lock<std::mutex>();
  const auto take = [&](size_t size) {
    if (!kept) return scratch(size, q);
    if (!kept->buffer.defined() || (size_t)kept->buffer.numel() < size || kept->buffer.device() != q.device()) {
      kept->listed.reset();
      kept->buffer.reset();
      kept->buffer = scratch(size, q);
    }
    return kept->buffer;
  };
  try {
    workspace = take(bytes);
  } catch (const c10::OutOfMemoryError&) {
    if (workspace_bytes >= 0 || bytes <= least || (form != 0 && !form_is_free)) throw;
    variant &= ~CT_ATTN_BWD_DQ_FROM_DS;
    bytes = least;
    workspace = take(bytes);
  }
  if (kept) {
    const bool versioned = !bounds.is_inference();
    auto wanted = std::make_tuple(versioned ? bounds.unsafeGetTensorImpl()->version_counter().current_version() : 0u,
                                  std::vector<int64_t>{s.batch, s.seq, s.q_heads, s.kv_heads, s.head_dim}, variant, bytes,
                                  (float)scale);
    if (versioned && kept->listed.is_same(bounds) && kept->listed_for == wanted) variant |= CT_ATTN_BWD_WORK_LIST_KEPT;
    kept->listed.reset();  // (until the call below has been made)
    kept->listed_for = std::move(wanted);
  }
  ct_attn_bwd_args a = {};
  a.q = bits(q);
  a.k = bits(k);
  a.v = bits(v);
  a.segment_ids = ptr<int32_t>(segments);
  a.attention_end = ptr<int32_t>(ends);
  a.tile_meta = ptr<int32_t>(bounds);
  a.out = bits(out);
  a.lse = ptr<float>(lse);
  a.dout = bits(dout);
  a.dq = bits(dq);
  a.dk = bits(dk);
  a.dv = bits(dv);
  a.delta = ptr<float>(delta);
  a.workspace = workspace.data_ptr();
  a.workspace_bytes = bytes;
  a.batch = s.batch;
  a.seq = s.seq;
  a.q_heads = s.q_heads;
  a.kv_heads = s.kv_heads;
  a.head_dim = s.head_dim;
  a.scale = (float)scale;
  a.variant = variant;
  check(ct_attn_bwd(current_stream(), &a));
  if (kept) kept->listed = bounds;
  return {dq, dk, dv, delta};
}

// The form of the backward that the operator asks for. Left open, the library takes dQ from stored dS blocks at
// rows of up to 4096 positions (what that gains and loses: beside the flag in ct_hotpath.h); longer ones ask for
// that form where it is the faster one and its workspace is at most 4 GiB. It saves the two products that the
// recomputing dQ kernel repeats and pays 2 KB written and read per block. Measured over rows of 4224 to 25600
// positions with documents from 16 positions to the whole row, recomputing / stored:
//   head dimension 128: 0.95 to 1.2, below 1 with documents of thousands of positions at up to 8000 row blocks only
//     ([3, 6144, 8/8 heads] documents of 16 to 64 112 / 95 us, of 64 to 6144 396 / 416, whole rows 728 / 734; [6, 10240, 8/8] 100 to
//     400 428 / 377, whole rows 3749 / 3662).
//   head dimension 64: a block's products are half as long and its traffic the same. Launches of few row blocks (32
//     query rows of one head) gain, up to 1400 of them ([1, 7424, 6/1], images, 159 / 115; [1, 5376, 6/2] 126 / 85); with 2048
//     whole-row documents lose (0.84 at [1, 16384, 4/1]), with 4096 most long ones (0.75 to 0.91).
int operator_form(const AttnShape& s, bool with_ends) {
  if (s.seq <= CT_ATTN_FROM_DS_UP_TO_SEQ) return 0;
  const bool pays = s.head_dim == 128 ? s.seq <= 32768
                                      : s.seq <= 8192 && (int64_t)s.batch * s.q_heads * (s.seq / 32) <= 1536;
  if (!pays) return 0;
  const size_t bytes = ct_attn_bwd_workspace_bytes_from_ds(s.batch, s.seq, s.q_heads, s.kv_heads, s.head_dim, with_ends);
  return bytes > 0 && bytes <= kFromDsWorkspaceCap ? CT_ATTN_BWD_DQ_FROM_DS : 0;
}

// The reference's residual (q, k, v, metadata, O, LSE) (src/causal_trainer/kernels/efficient_attention.py:1831-1863)
struct AttentionNode : OperatorNode {
  SavedVariable q, k, v, out, lse;
  Tensor segments, bounds;
  MaybeTensor ends;
  double scale = 0;
  std::shared_ptr<KeptWorkspace> kept;

  variable_list differentiate(variable_list&& grads) override {
    const auto self = shared_from_this();
    const Tensor Q = q.unpack(), K = k.unpack(), V = v.unpack(), O = out.unpack(self), L = lse.unpack();
    auto [dq, dk, dv, delta] =
        attention_backward(Q, K, V, segments, ends, bounds, O, L, gradient(grads[0], O.sizes(), at::kBFloat16, O), scale,
                           operator_form(attn_shape(Q, K), ends && ends->defined()), -1, kept.get(), true);
    return {dq, dk, dv};
  }
  void release_variables() override {
    q.reset_data();
    k.reset_data();
    v.reset_data();
    out.reset_data();
    lse.reset_data();
  }
  std::string name() const override { return "EfficientAttentionBackward"; }
};

MaybeTensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& query_ids, const Tensor& key_ids,
                      const Tensor& q_blocks, const Tensor& kv_blocks, const MaybeTensor& ends, const MaybeTensor& bounds,
                      int64_t block_q, int64_t block_kv, double scale, const std::shared_ptr<KeptWorkspace>& kept) {
  if (!plain(q, at::kBFloat16, 4) || !plain(k, at::kBFloat16, 4) || !plain(v, at::kBFloat16, 4) || !std::isfinite(scale))
    return std::nullopt;
  const int64_t batch = q.size(0), seq = q.size(1), dim = q.size(3);
  for (const Tensor& t : {k, v, query_ids})
    if (t.device() != q.device()) return std::nullopt;
  if (k.sizes() != v.sizes() || k.size(0) != batch || k.size(1) != seq || k.size(3) != dim || (dim != 64 && dim != 128) ||
      q.numel() == 0 || k.numel() == 0 || q.size(2) % k.size(2))
    return std::nullopt;
  const int64_t ids_shape[2] = {batch, seq};
  const at::IntArrayRef ids(ids_shape, 2);
  const bool hybrid = ends && ends->defined();
  if (!bounds || !bounds->defined() || !plain(query_ids, at::kInt, 2) || query_ids.sizes() != ids ||
      !plain(key_ids, at::kInt, 2) || key_ids.sizes() != ids || !plain(q_blocks, at::kInt, 3) ||
      q_blocks.sizes() != at::IntArrayRef({batch, seq / block_q, hybrid ? 3 : 2}) || !plain(kv_blocks, at::kInt, 3) ||
      kv_blocks.sizes() != at::IntArrayRef({batch, seq / block_kv, 2}) ||
      (hybrid && (!plain(*ends, at::kInt, 2) || ends->sizes() != ids)) || !plain(*bounds, at::kInt, 1) ||
      (size_t)bounds->numel() * 4 != ct_attn_meta_bytes((int32_t)batch, (int32_t)seq))
    return std::nullopt;
  auto [out, lse] = attention_forward(q, k, v, query_ids, ends, *bounds, scale);
  if (needs_graph({q, k, v})) {
    auto node = graph_node<AttentionNode>({q, k, v});
    node->q = SavedVariable(q, false);
    node->k = SavedVariable(k, false);
    node->v = SavedVariable(v, false);
    node->lse = SavedVariable(lse, false);
    node->segments = query_ids;
    node->ends = ends;
    node->bounds = *bounds;
    node->scale = scale;
    node->kept = kept;
    torch::autograd::set_history(out, node);
    node->out = SavedVariable(out, true);
  }
  return out;
}

// ---------------------------------------------------------------------------------------------
// RMS norm and rotary embedding
// ---------------------------------------------------------------------------------------------
struct RmsNormNode : OperatorNode {
  SavedVariable x, scale;
  // Of few rows, 4 KB at most. Beside the residuals: what saved-tensor hooks are given stays x and scale, for any number of rows
  // (x is unpacked first, so that a graph that was released or an x that was overwritten is refused as before).
  Tensor rstd;
  double eps = 0;
  variable_list differentiate(variable_list&& grads) override {
    const Tensor X = x.unpack(), W = scale.unpack();
    const c10::DeviceGuard guard(X.device());
    const int64_t hidden = X.size(-1), rows = X.numel() / hidden;
    const Tensor dy = gradient(grads[0], X.sizes(), at::kBFloat16, X);
    Tensor dx = fresh(X), dscale = fresh(W);
    if (rstd.defined()) {
      check(ct_rms_norm_bwd_saved(current_stream(), bits(X), bits(W), bits(dy), ptr<float>(rstd), rows, (int32_t)hidden, bits(dx),
                                  bits(dscale)));
      return {dx, dscale};
    }
    const size_t bytes = ct_rms_norm_bwd_workspace_bytes((int32_t)hidden);
    Tensor workspace = scratch(bytes, X);
    check(ct_rms_norm_bwd_rounded(current_stream(), bits(X), bits(W), bits(dy), (float)eps, rows, (int32_t)hidden, bits(dx),
                                  bits(dscale), workspace.data_ptr(), bytes));
    return {dx, dscale};
  }
  void release_variables() override {
    x.reset_data();
    scale.reset_data();
    rstd.reset();
  }
  std::string name() const override { return "RmsNormBackward"; }
};

MaybeTensor rms_norm(const Tensor& x, const Tensor& scale, double eps) {
  if (x.dim() == 0 || !plain(x, at::kBFloat16, x.dim()) || !plain(scale, at::kBFloat16, 1) || scale.device() != x.device() ||
      scale.size(0) != x.size(-1) || x.numel() == 0)
    return std::nullopt;
  const c10::DeviceGuard guard(x.device());
  const int64_t hidden = x.size(-1), rows = x.numel() / hidden;
  const bool graph = needs_graph({x, scale});
  Tensor y = fresh(x), rstd;
  if (graph && ct_rms_norm_keeps_rstd(rows, (int32_t)hidden)) rstd = floats({rows}, x);
  check(ct_rms_norm_fwd(current_stream(), bits(x), bits(scale), (float)eps, rows, (int32_t)hidden, bits(y),
                        rstd.defined() ? ptr<float>(rstd) : nullptr));
  if (graph) {
    auto node = graph_node<RmsNormNode>({x, scale});
    node->x = SavedVariable(x, false);
    node->scale = SavedVariable(scale, false);
    node->rstd = rstd;
    node->eps = eps;
    torch::autograd::set_history(y, node);
  }
  return y;
}

std::tuple<Tensor, Tensor> rotate(const Tensor& q, const Tensor& k, const Tensor& cosine, const Tensor& sine, int style,
                                  bool inverse, double q_scale) {
  const c10::DeviceGuard guard(q.device());
  Tensor q_out = fresh(q), k_out = fresh(k);
  ct_rotary_args a = {};
  a.q_in = bits(q);
  a.k_in = bits(k);
  a.q_out = bits(q_out);
  a.k_out = bits(k_out);
  a.cosine = bits(cosine);
  a.sine = bits(sine);
  a.tokens = q.size(0) * q.size(1);
  a.q_heads = (int32_t)q.size(2);
  a.kv_heads = (int32_t)k.size(2);
  a.head_dim = (int32_t)q.size(3);
  a.rotary_pairs = (int32_t)cosine.size(-1);
  a.rope_style = style;
  a.inverse = inverse ? 1 : 0;
  a.q_scale = (float)q_scale;
  check(ct_apply_rotary(current_stream(), &a));
  return {q_out, k_out};
}

struct RotaryNode : OperatorNode {
  SavedVariable cosine, sine;
  std::vector<int64_t> q_shape, k_shape;
  int style = 0;
  double q_scale = 1;
  variable_list differentiate(variable_list&& grads) override {
    const Tensor C = cosine.unpack(), S = sine.unpack();
    const Tensor dq = gradient(grads[0], q_shape, at::kBFloat16, C), dk = gradient(grads[1], k_shape, at::kBFloat16, C);
    auto [q, k] = rotate(dq, dk, C, S, style, true, q_scale);
    return {q, k};
  }
  void release_variables() override {
    cosine.reset_data();
    sine.reset_data();
  }
  std::string name() const override { return "ApplyRotaryBackward"; }
};

std::optional<std::tuple<Tensor, Tensor>> apply_rotary(const Tensor& q, const Tensor& k, const Tensor& cosine,
                                                       const Tensor& sine, int style, double q_scale) {
  if (!plain(q, at::kBFloat16, 4) || !plain(k, at::kBFloat16, 4) || !plain(cosine, at::kBFloat16, 3) ||
      !plain(sine, at::kBFloat16, 3) || q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(3) != k.size(3) ||
      cosine.sizes() != sine.sizes() || cosine.size(0) != q.size(0) || cosine.size(1) != q.size(1) || q.numel() == 0 ||
      k.numel() == 0 || cosine.size(2) == 0 || 2 * cosine.size(2) > q.size(3))
    return std::nullopt;
  auto [q_out, k_out] = rotate(q, k, cosine, sine, style, false, q_scale);
  if (needs_graph({q, k})) {
    auto node = graph_node<RotaryNode>({q, k});
    node->cosine = SavedVariable(cosine, false);
    node->sine = SavedVariable(sine, false);
    node->q_shape = q.sizes().vec();
    node->k_shape = k.sizes().vec();
    node->style = style;
    node->q_scale = q_scale;
    torch::autograd::set_history(q_out, node);
    torch::autograd::set_history(k_out, node);
  }
  return std::make_tuple(q_out, k_out);
}

// ---------------------------------------------------------------------------------------------
// cross-entropy
// ---------------------------------------------------------------------------------------------
constexpr int32_t kIgnoreIndex = -100;

ct_sparse_ce_args sparse_args(const Tensor& logits, const Tensor& targets, const Tensor& weights) {
  ct_sparse_ce_args a = {};
  a.logits = logits.data_ptr();
  a.targets = ptr<int32_t>(targets);
  a.weights = ptr<float>(weights);
  a.vocab = (int32_t)logits.size(-1);
  a.rows = logits.numel() / logits.size(-1);
  a.logits_dtype = logits.scalar_type() == at::kFloat ? CT_DTYPE_F32 : CT_DTYPE_BF16;
  a.ignore_index = kIgnoreIndex;
  return a;
}

struct SparseCeNode : OperatorNode {
  SavedVariable logits, targets, weights, lse;
  variable_list differentiate(variable_list&& grads) override {
    const Tensor X = logits.unpack(), T = targets.unpack(), W = weights.unpack(), L = lse.unpack();
    const c10::DeviceGuard guard(X.device());
    const Tensor dy = gradient(grads[0], T.sizes(), at::kFloat, X);
    Tensor dlogits = fresh(X);
    const ct_sparse_ce_args a = sparse_args(X, T, W);
    check(ct_sparse_ce_bwd(current_stream(), &a, ptr<float>(L), ptr<float>(dy), dlogits.data_ptr()));
    return {dlogits};
  }
  void release_variables() override {
    logits.reset_data();
    targets.reset_data();
    weights.reset_data();
    lse.reset_data();
  }
  std::string name() const override { return "SparseCrossEntropyBackward"; }
};

MaybeTensor sparse_ce(const Tensor& logits, const Tensor& targets, const Tensor& weights) {
  if (logits.dim() != 3 || (!plain(logits, at::kBFloat16, 3) && !plain(logits, at::kFloat, 3)) || logits.numel() == 0 ||
      !plain(targets, at::kInt, 2) || !plain(weights, at::kFloat, 2) || targets.sizes() != logits.sizes().slice(0, 2) ||
      weights.sizes() != targets.sizes() || targets.device() != logits.device() || weights.device() != logits.device())
    return std::nullopt;
  const c10::DeviceGuard guard(logits.device());
  Tensor loss = floats(targets.sizes(), logits), lse = floats(targets.sizes(), logits);
  const ct_sparse_ce_args a = sparse_args(logits, targets, weights);
  check(ct_sparse_ce_fwd(current_stream(), &a, ptr<float>(loss), ptr<float>(lse)));
  if (needs_graph({logits})) {
    auto node = graph_node<SparseCeNode>({logits});
    node->logits = SavedVariable(logits, false);
    node->targets = SavedVariable(targets, false);
    node->weights = SavedVariable(weights, false);
    node->lse = SavedVariable(lse, false);
    torch::autograd::set_history(loss, node);
  }
  return loss;
}

// hidden [..., d], head [d, V], targets / weights one per row of hidden
ct_cutce_shape cut_shape(const Tensor& hidden, const Tensor& head) {
  const int64_t width = hidden.size(-1);
  return {(int32_t)(hidden.numel() / width), (int32_t)width, (int32_t)head.size(1)};
}

// head: [d, V], or the panel itself (then read from there only)
std::tuple<Tensor, Tensor, Tensor> cutce_forward_on(const ct_cutce_shape& shape, const Tensor& hidden, const Tensor& head,
                                                    const Tensor& targets, const Tensor& weights, bool compaction,
                                                    const MaybeTensor& cache, int64_t workspace_bytes, const MaybeTensor& panel,
                                                    bool filled) {
  const c10::DeviceGuard guard(hidden.device());
  // (with a logits cache the aligned copy of an unaligned head goes there)
  const bool cached = cache && cache->defined();
  const size_t bytes = cached || panel ? ct_cutce_fwd_workspace_min_bytes(&shape)
                       : workspace_bytes >= 0 ? (size_t)workspace_bytes : ct_cutce_fwd_workspace_used_bytes(&shape);
  Tensor workspace = scratch(bytes, hidden);
  Tensor nll = floats({}, hidden), weight_sum = floats({}, hidden), lse = floats({shape.rows}, hidden);
  ct_cutce_fwd_args a = {};
  a.hidden = bits(hidden);
  a.head = bits(head);
  a.targets = ptr<int32_t>(targets);
  a.weights = ptr<float>(weights);
  a.nll_sum = ptr<float>(nll);
  a.weight_sum = ptr<float>(weight_sum);
  a.lse = ptr<float>(lse);
  a.workspace = workspace.data_ptr();
  a.workspace_bytes = bytes;
  a.shape = shape;
  a.sparse_compaction = compaction;
  a.logits_cache = cached ? cache->data_ptr() : nullptr;
  a.logits_cache_bytes = cached ? (size_t)cache->numel() : 0;
  check(ct_cutce_fwd_panel(current_stream(), &a, panel ? bits(*panel) : nullptr, panel ? panel->nbytes() : 0, filled));
  return {nll, weight_sum, lse};
}
std::tuple<Tensor, Tensor, Tensor> cutce_forward(const Tensor& hidden, const Tensor& head, const Tensor& targets,
                                                 const Tensor& weights, bool compaction, const MaybeTensor& cache,
                                                 int64_t workspace_bytes) {
  return cutce_forward_on(cut_shape(hidden, head), hidden, head, targets, weights, compaction, cache, workspace_bytes,
                          std::nullopt, false);
}

std::tuple<Tensor, MaybeTensor> cutce_backward_on(const ct_cutce_shape& shape, const Tensor& hidden, const Tensor& head,
                                                  const Tensor& targets, const Tensor& weights, const Tensor& lse,
                                                  const Tensor& dy, bool compaction, bool with_head, int64_t workspace_bytes,
                                                  const MaybeTensor& cache, const MaybeTensor& panel) {
  const c10::DeviceGuard guard(hidden.device());
  const bool cached = cache && cache->defined();
  const size_t bytes = workspace_bytes >= 0 ? (size_t)workspace_bytes
                       : cached || panel    ? ct_cutce_bwd_workspace_bytes(&shape) - ct_cutce_panel_bytes(&shape)
                                            : ct_cutce_bwd_workspace_used_bytes(&shape);
  Tensor workspace = scratch(bytes, hidden), dhidden = fresh(hidden);
  MaybeTensor dhead;
  if (with_head) dhead = at::empty({shape.hidden, shape.vocab}, hidden.options().requires_grad(false));
  ct_cutce_bwd_args a = {};
  a.hidden = bits(hidden);
  a.head = bits(head);
  a.targets = ptr<int32_t>(targets);
  a.weights = ptr<float>(weights);
  a.lse = ptr<float>(lse);
  a.dy = ptr<float>(dy);
  a.dhidden = bits(dhidden);
  a.dhead = dhead ? bits(*dhead) : nullptr;
  a.workspace = workspace.data_ptr();
  a.workspace_bytes = bytes;
  a.shape = shape;
  a.sparse_compaction = compaction;
  a.logits_cache = cached ? cache->data_ptr() : nullptr;
  a.logits_cache_bytes = cached ? (size_t)cache->numel() : 0;
  check(ct_cutce_bwd_panel(current_stream(), &a, panel ? bits(*panel) : nullptr, panel ? panel->nbytes() : 0));
  return {dhidden, dhead};
}
std::tuple<Tensor, MaybeTensor> cutce_backward(const Tensor& hidden, const Tensor& head, const Tensor& targets,
                                               const Tensor& weights, const Tensor& lse, const Tensor& dy, bool compaction,
                                               bool with_head, int64_t workspace_bytes, const MaybeTensor& cache) {
  return cutce_backward_on(cut_shape(hidden, head), hidden, head, targets, weights, lse, dy, compaction, with_head,
                           workspace_bytes, cache, std::nullopt);
}

// The reference's residual (src/causal_trainer/kernels/cut_cross_entropy.py:587-593), for a [V, d] head with its transposed
// copy (a panel where the vocabulary is unaligned) in the head's place. Where the caller lets the operator keep more
// than that (use_cache), one of two buffers that the first backward gives back: the f32 logits cache, or the panel that
// the forward has read an unaligned head from.
struct CutCeNode : OperatorNode {
  SavedVariable hidden, head, targets, weights, lse;
  MaybeTensor cache, panel;
  ct_cutce_shape shape = {};
  bool head_is_panel = false;
  bool compaction = false, trainable = true, vocab_major = false;
  int64_t workspace_bytes = -1;
  variable_list differentiate(variable_list&& grads) override {
    const Tensor X = hidden.unpack(), W = head.unpack(), T = targets.unpack(), w = weights.unpack(), L = lse.unpack();
    const Tensor dy = gradient(grads[0], {}, at::kFloat, X);
    const MaybeTensor logits = std::exchange(cache, std::nullopt), copy = std::exchange(panel, std::nullopt);
    auto [dx, dw] = cutce_backward_on(shape, X, W, T, w, L, dy, compaction, trainable, workspace_bytes, logits,
                                      head_is_panel ? MaybeTensor(W) : copy);
    return {dx, !dw ? Tensor() : vocab_major ? dw->t() : *dw};
  }
  void release_variables() override {
    hidden.reset_data();
    head.reset_data();
    targets.reset_data();
    weights.reset_data();
    lse.reset_data();
    cache.reset();
    panel.reset();
  }
  std::string name() const override { return "CutCrossEntropyBackward"; }
};

// The logits cache pays where it saves more than it costs: 8 bytes of traffic per logit and a pass of its
// own against 2 * hidden operations. Measured with and without it (train step, us): 4096 rows x 32000, hidden
// 768: 815 / 782, 896: 885 / 876, 1024: 916 / 928, 1280: 1081 / 1128; 800 x 151936, 768: 929 / 917, 1024: 1110 / 1163;
// 16384 x 50000, 896: 5553 / 5748. Logits that stay in the memory-side cache (256 MB) cost no less: 1000 x 32003, 512:
// 208 / 187, 768: 261 / 255, 1024: 300 / 317; 2000 x 20000, 256: 187 / 159; 3000 x 16000, 512: 266 / 234, 640: 315 / 305;
// 4096 x 3200, 512: 113 / 114, 1024: 147 / 159; 130 x 76000, 512: 163 / 165.
bool cache_pays(const ct_cutce_shape& shape) { return shape.hidden > 768; }

// The largest panel that is kept. Train steps, us, panel kept / made by each direction: 1000 rows x 32003, hidden 512: 192 / 199,
// 768: 256 / 263; 300 x 105349, 256: 240 / 252; 4096 x 50257, 768: 1094 / 1136; 50 x 74295, 768: 246 / 285.
constexpr int64_t kPanelLimit = (int64_t)1 << 30;

// vocab_major: head is [V, d]; the kernels get a transposed copy, the gradient goes back as a view of theirs.
std::optional<std::tuple<Tensor, Tensor>> cut_ce(const Tensor& hidden, const Tensor& head, const Tensor& targets,
                                                 const Tensor& weights, bool trainable, bool compaction, bool use_cache,
                                                 int64_t cache_limit, int64_t forward_bytes, int64_t backward_bytes,
                                                 bool vocab_major) {
  if (!plain(hidden, at::kBFloat16, 3) || !plain(head, at::kBFloat16, 2) || !plain(targets, at::kInt, 2) ||
      !plain(weights, at::kFloat, 2) || hidden.numel() == 0 || head.numel() == 0 || hidden.size(2) % 128 ||
      head.size(vocab_major ? 1 : 0) != hidden.size(2) || targets.sizes() != hidden.sizes().slice(0, 2) ||
      weights.sizes() != targets.sizes() || head.device() != hidden.device() || targets.device() != hidden.device() ||
      weights.device() != hidden.device())
    return std::nullopt;
  const bool graph = needs_graph({hidden, head});
  const int64_t width = hidden.size(2);
  const ct_cutce_shape shape = {(int32_t)(hidden.numel() / width), (int32_t)width, (int32_t)head.size(vocab_major ? 0 : 1)};
  const c10::DeviceGuard guard(head.device());
  // (A bounded workspace: the copies keep to it. A [V, d] head is otherwise transposed straight into a panel: [35263, 7552] and
  // 21 rows 1366 -> 875 us, its plain transposed copy was copied again by each direction.)
  const size_t panel_bytes = forward_bytes < 0 ? ct_cutce_panel_bytes(&shape) : 0;
  const bool head_is_panel = vocab_major && panel_bytes;
  Tensor columns = head;  // [d, V], padded in a panel
  if (vocab_major) {
    const int64_t ld = head_is_panel ? (int64_t)(panel_bytes / 2) / width : shape.vocab;
    columns = at::empty({width, ld}, head.options().requires_grad(false));
    check(ct_transpose16_padded(current_stream(), bits(head), shape.vocab, shape.hidden, bits(columns), (int32_t)ld));
  }
  MaybeTensor cache, panel;
  if (use_cache && graph) {
    const size_t bytes = head_is_panel ? ct_cutce_logits_cache_bytes(&shape) - panel_bytes : ct_cutce_logits_cache_used_bytes(&shape);
    if ((int64_t)bytes <= cache_limit && cache_pays(shape)) cache = scratch(bytes, hidden);
  }
  // An unaligned head is copied once for both directions only where the caller lets a buffer be kept between them, like
  // the logits cache, which holds such a copy itself. Otherwise each direction makes one in its workspace or reads it in
  // place; with few rows both do.
  if (head_is_panel) panel = columns;
  else if (use_cache && graph && !cache && panel_bytes && (int64_t)panel_bytes <= std::min(kPanelLimit, cache_limit) &&
           !ct_cutce_head_in_place(&shape))
    panel = scratch(panel_bytes, hidden);
  auto [nll, weight_sum, lse] =
      cutce_forward_on(shape, hidden, columns, targets, weights, compaction, cache, forward_bytes, panel, head_is_panel);
  if (graph) {
    auto node = graph_node<CutCeNode>({hidden, head});
    node->hidden = SavedVariable(hidden, false);
    node->head = SavedVariable(columns, false);
    node->shape = shape;
    node->head_is_panel = head_is_panel;
    if (!head_is_panel) node->panel = panel;
    node->targets = SavedVariable(targets, false);
    node->weights = SavedVariable(weights, false);
    node->lse = SavedVariable(lse, false);
    node->cache = cache;
    node->compaction = compaction;
    node->trainable = trainable;
    node->vocab_major = vocab_major;
    node->workspace_bytes = backward_bytes;
    torch::autograd::set_history(nll, node);
  }
  return std::make_tuple(nll, weight_sum);
}

// ---------------------------------------------------------------------------------------------
// preparation of a batch
// ---------------------------------------------------------------------------------------------
MaybeTensor canonical_ids(const Tensor& mask, const MaybeTensor& labels) {
  if (!plain(mask, at::kInt, 2) || mask.numel() == 0 || (labels && (!plain(*labels, at::kInt, 2) || labels->sizes() != mask.sizes())))
    return std::nullopt;
  const c10::DeviceGuard guard(mask.device());
  Tensor out = ints(mask.sizes(), mask);
  check(ct_canonicalize_segment_ids(current_stream(), ptr<int32_t>(mask), ptr<int32_t>(labels), (int32_t)mask.size(0),
                                    (int32_t)mask.size(1), ptr<int32_t>(out)));
  return out;
}

// positions inside the runs of (mask, labels)
MaybeTensor segment_positions(const Tensor& mask, const MaybeTensor& labels) {
  if (!plain(mask, at::kInt, 2) || mask.numel() == 0 || (labels && (!plain(*labels, at::kInt, 2) || labels->sizes() != mask.sizes())))
    return std::nullopt;
  const c10::DeviceGuard guard(mask.device());
  Tensor out = ints(mask.sizes(), mask);
  check(ct_segment_positions(current_stream(), ptr<int32_t>(mask), ptr<int32_t>(labels), (int32_t)mask.size(0),
                             (int32_t)mask.size(1), ptr<int32_t>(out)));
  return out;
}

std::optional<std::tuple<Tensor, Tensor>> rotary_tables(const Tensor& positions, const Tensor& inv_freq) {
  if (!plain(positions, at::kInt, 2) || !plain(inv_freq, at::kFloat, 1) || positions.numel() == 0 || inv_freq.numel() == 0 ||
      inv_freq.device() != positions.device())
    return std::nullopt;
  const c10::DeviceGuard guard(positions.device());
  const int64_t pairs = inv_freq.numel();
  const auto options = positions.options().dtype(at::kBFloat16);
  Tensor cosine = at::empty({positions.size(0), positions.size(1), pairs}, options);
  Tensor sine = at::empty({positions.size(0), positions.size(1), pairs}, options);
  check(ct_rotary_cos_sin(current_stream(), ptr<int32_t>(positions), ptr<float>(inv_freq), positions.numel(), (int32_t)pairs,
                          bits(cosine), bits(sine)));
  return std::make_tuple(cosine, sine);
}

std::optional<std::tuple<Tensor, Tensor>> shifted_targets(const Tensor& tokens, const MaybeTensor& mask,
                                                          const MaybeTensor& segments, const MaybeTensor& assistant,
                                                          const MaybeTensor& loss_mask, const MaybeTensor& labels,
                                                          int64_t ignore_index) {
  if (!plain(tokens, at::kInt, 2) || tokens.size(0) == 0 || tokens.size(1) < 2) return std::nullopt;
  for (const MaybeTensor* t : {&mask, &segments, &assistant, &labels})
    if (*t && (!plain(**t, at::kInt, 2) || (*t)->sizes() != tokens.sizes())) return std::nullopt;
  if (loss_mask && (!plain(*loss_mask, at::kFloat, 2) || loss_mask->sizes() != tokens.sizes())) return std::nullopt;
  const c10::DeviceGuard guard(tokens.device());
  const int64_t batch = tokens.size(0), seq = tokens.size(1);
  Tensor targets = ints({batch, seq - 1}, tokens), weights = floats({batch, seq - 1}, tokens);
  ct_shifted_targets_args a = {};
  a.input_ids = ptr<int32_t>(tokens);
  a.attention_mask = ptr<int32_t>(mask);
  a.segment_ids = ptr<int32_t>(segments);
  a.assistant_mask = ptr<int32_t>(assistant);
  a.loss_mask = ptr<float>(loss_mask);
  a.labels = ptr<int32_t>(labels);
  a.targets = ptr<int32_t>(targets);
  a.weights = ptr<float>(weights);
  a.batch = (int32_t)batch;
  a.seq = (int32_t)seq;
  a.ignore_index = (int32_t)ignore_index;
  check(ct_shifted_targets_and_weights(current_stream(), &a));
  return std::make_tuple(targets, weights);
}

// (tile bounds, query summary, key summary, whether a graph's replays will write them); segment ids and ends
// already int32, contiguous, on the GPU
std::tuple<Tensor, Tensor, Tensor, bool> attention_metadata(const Tensor& segments, const MaybeTensor& ends,
                                                            int64_t block_q, int64_t block_kv) {
  const c10::DeviceGuard guard(segments.device());
  const int32_t batch = (int32_t)segments.size(0), seq = (int32_t)segments.size(1);
  Tensor bounds = ints({(int64_t)(ct_attn_meta_bytes(batch, seq) / 4)}, segments);
  Tensor q_summary = ints({batch, seq / block_q, ends ? 3 : 2}, segments), kv_summary = ints({batch, seq / block_kv, 2}, segments);
  void* stream = current_stream();
  if (block_q % 32 == 0 && block_kv % 32 == 0) {
    check(ct_attn_prepare_summaries(stream, ptr<int32_t>(segments), ptr<int32_t>(ends), batch, seq, ptr<int32_t>(bounds),
                                    (int32_t)block_q, ptr<int32_t>(q_summary), (int32_t)block_kv, ptr<int32_t>(kv_summary)));
    return {bounds, q_summary, kv_summary, capturing()};
  }
  check(ct_attn_prepare(stream, ptr<int32_t>(segments), ptr<int32_t>(ends), batch, seq, ptr<int32_t>(bounds)));
  check(ct_attn_block_summary(stream, ptr<int32_t>(segments), ptr<int32_t>(ends), batch, seq, (int32_t)block_q,
                              ptr<int32_t>(q_summary)));
  check(ct_attn_block_summary(stream, ptr<int32_t>(segments), nullptr, batch, seq, (int32_t)block_kv, ptr<int32_t>(kv_summary)));
  return {bounds, q_summary, kv_summary, capturing()};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_error_class", [](py::object cls) { error_class = cls.release(); });
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const StatusError& e) {
      set_python_error(e);
    }
  });
  py::class_<KeptWorkspace, std::shared_ptr<KeptWorkspace>>(m, "KeptWorkspace").def(py::init<>());
  // The GIL is only needed to convert arguments and results: allocations and launches may block.
  const auto def = [&m](const char* name, auto function) { m.def(name, function, py::call_guard<py::gil_scoped_release>()); };
  def("attention", &attention);
  def("attention_forward", &attention_forward);
  def("attention_backward", &attention_backward);
  def("rms_norm", &rms_norm);
  def("apply_rotary", &apply_rotary);
  def("sparse_ce", &sparse_ce);
  def("cut_ce", &cut_ce);
  def("cutce_forward", &cutce_forward);
  def("cutce_backward", &cutce_backward);
  def("canonical_ids", &canonical_ids);
  def("segment_positions", &segment_positions);
  def("rotary_tables", &rotary_tables);
  def("shifted_targets", &shifted_targets);
  def("attention_metadata", &attention_metadata);
}
