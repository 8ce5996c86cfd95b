"""Host-side mirror of the reference's Cut cross-entropy operator for MI355X.

``pallas_cut_linear_cross_entropy`` keeps the reference's name, argument
meaning, validation errors and custom-VJP contract
(src/causal_trainer/kernels/cut_cross_entropy.py:828-958, :524-670): it
returns ``(nll_sum, weight_sum)`` as f32 scalars, saves
``(hidden, head, targets, weights, lse)``, gives no cotangent to
targets / weights, ignores the cotangent of ``weight_sum``, and with
``lm_head_trainable=False`` never launches the dHead kernel and returns no
head gradient. Tensors are torch tensors on a ROCm device; the work is done by
libct_hotpath.so through its C ABI.

``loss = nll_sum / max(weight_sum, 1)`` stays with the caller
(src/causal_trainer/training/losses.py:234-237).

One deliberate difference in the residual. The reference keeps no logits because
a TPU core has little memory, and pays for it by recomputing the projection in
each backward kernel. A MI355X has 288 GB: when the f32 logits of the active
rows fit in ``LOGITS_CACHE_LIMIT_BYTES`` the forward also leaves them in a cache
that lives until the backward of the loss (the adjacent step of a training
iteration), and the backward then runs 3 GEMMs instead of 4. Above the limit, or where
the projection is cheaper than the cache's traffic (small hidden sizes), the logits are
recomputed, and what is kept in the cache's place is the aligned copy that a head whose
vocabulary is no multiple of 8 is read through, up to the limit and 1 GiB (with few rows such a head is read
in place, and nothing is kept). Like the cache it
is no saved tensor (hooks do not see it) and goes with the first backward. With
``logits_cache=False`` nothing but ``lse`` is kept: logits and copy are made again.

``local_chunk_size`` (:697-825). The reference's chunk loop bounds what one TPU core holds at
a time: it walks the rows in chunks, compacts inside the chunk and accumulates the head
gradient in f32 across chunks. What the option buys is a bound on transient memory, and that
is what it selects here: with ``local_chunk_size = C > 0`` the backward's workspace is the share
C / rows of what a single slab over the whole vocabulary takes with the aligned copy of an unaligned
head (``backward_workspace_bytes``; never below the kernels' minimum of one 256-wide vocabulary tile,
and where the head is read in place no more than the slab without the copy), the vocabulary is walked in
slabs that fit with dHidden accumulated in f32 across slabs and rounded once, and no logits
cache is kept. A row's statistics and gradients do not depend on which slab or slot it sits in;
only the order of f32 additions differs, inside the operator's tolerances. ``0`` (the default)
keeps the single full-vocabulary slab.
"""

from __future__ import annotations

import functools

import torch

from . import _lib
from .efficient_attention import _Axes, _integer

_HIDDEN_ALIGN = 128
# Largest logits cache the operator allocates by itself (f32 [vocab, rows], both padded to 256).
LOGITS_CACHE_LIMIT_BYTES = 24 << 30


def _shape_struct(rows: int, hidden: int, vocab: int) -> _lib.CutceShape:
    return _lib.CutceShape(rows=rows, hidden=hidden, vocab=vocab)


def logits_cache_bytes(rows: int, hidden: int, vocab: int) -> int:
    """Size of the optional f32 logits cache for this problem."""

    return int(_lib.load().ct_cutce_logits_cache_used_bytes(_shape_struct(rows, hidden, vocab)))


def backward_workspace_bytes(rows: int, hidden: int, vocab: int, local_chunk_size: int = 0) -> int:
    """Workspace of the backward: what the full-vocabulary slab uses, or with ``local_chunk_size`` rows per chunk their
    share of that slab and a copy of the head (at least the kernels' minimum)."""

    lib = _lib.load()
    shape = _shape_struct(rows, hidden, vocab)
    most, least = int(lib.ct_cutce_bwd_workspace_used_bytes(shape)), int(lib.ct_cutce_bwd_workspace_min_bytes(shape))
    if local_chunk_size <= 0 or local_chunk_size >= rows:
        return most
    full = int(lib.ct_cutce_bwd_workspace_bytes(shape))
    return max(least, min(most, least + (full - least) * local_chunk_size // rows))


def cutce_forward(hidden, head, targets, weights, *, sparse_compaction: bool = False,
                  logits_cache=None):
    """Flat forward: hidden [N, d], head [d, V] -> (nll_sum, weight_sum, lse [N]).

    ``logits_cache``: optional uint8 device tensor of ``logits_cache_bytes(...)`` bytes that
    the forward fills for ``cutce_backward``.
    """

    return _lib.native().cutce_forward(hidden.detach(), head.detach(), targets, weights, bool(sparse_compaction),
                                       logits_cache, -1)


def cutce_backward(hidden, head, targets, weights, lse, dy, *, sparse_compaction: bool = False,
                   lm_head_trainable: bool = True, workspace_bytes: int | None = None,
                   logits_cache=None):
    """Flat backward: returns (dhidden [N, d], dhead [d, V] or None).

    ``logits_cache``: the tensor a forward with the same ``sparse_compaction`` filled, or None
    to recompute the logits.
    """

    dy = dy.to(device=hidden.device, dtype=torch.float32).reshape(1).contiguous()
    return _lib.native().cutce_backward(
        hidden.detach(), head.detach(), targets, weights, lse, dy, bool(sparse_compaction), bool(lm_head_trainable),
        -1 if workspace_bytes is None else int(workspace_bytes), logits_cache)


@functools.lru_cache(maxsize=256)
def _workspaces(rows: int, hidden: int, vocab: int, local_chunk_size: int):
    """(forward, backward) workspace sizes; -1 leaves the choice to the library."""

    if local_chunk_size <= 0:
        return -1, -1
    backward = backward_workspace_bytes(rows, hidden, vocab, local_chunk_size)
    lib, shape = _lib.load(), _shape_struct(rows, hidden, vocab)
    # (the forward's part that may be smaller, an aligned copy of the head, keeps to the same bound)
    forward = max(lib.ct_cutce_fwd_workspace_min_bytes(shape), min(lib.ct_cutce_fwd_workspace_used_bytes(shape), backward))
    return int(forward), int(backward)


def _cut(hidden, head, targets, weights, trainable, cache, chunk, layout):
    """The operator on plain arguments (what the native side checks), None for any other."""

    try:
        if targets.shape != weights.shape or hidden.shape[:-1] != targets.shape:
            return None
        rows, width, vocab = targets.numel(), hidden.shape[-1], head.shape[layout == "dv"]
        if rows == 0 or width == 0 or vocab == 0:
            return None
        sizes = (-1, -1) if chunk == 0 else _workspaces(rows, width, vocab, chunk)
        return _lib.native().cut_ce(hidden, head, targets, weights, bool(trainable), True,
                                    bool(cache) and chunk == 0, LOGITS_CACHE_LIMIT_BYTES, *sizes, layout == "vd")
    except (AttributeError, IndexError, TypeError):
        return None     # (something is wrong with the arguments: the validation says what)


def pallas_cut_linear_cross_entropy(hidden_states, lm_head_kernel, targets, weights, *, mesh=None,
                                    sparse_compaction: bool = False,
                                    lm_head_trainable: bool = True, local_chunk_size: int = 0,
                                    logits_cache: bool = True, head_layout: str = "dv"):
    """Return ``(nll_sum, weight_sum)``; logits are only ever kept in the bounded cache
    described in the module docstring, which also says what is kept where it does not pay
    (``logits_cache=False``: nothing but the residuals of the module docstring's first paragraph).

    hidden_states ``[B, S, d]``, lm_head_kernel ``[d, V]`` (same float dtype, bf16),
    targets int32 ``[B, S]``, weights f32 ``[B, S]``; a row is ignored iff its weight is 0.

    ``sparse_compaction`` is a choice of speed in the reference and leaves the results alone; here ignored rows
    are left out of the products with either value. The kernels gather rows while they copy tiles, so that
    costs nothing: with no row ignored 0 to 4 us a pass more than rows in place (4096 x 32000, hidden 1024: 932
    against 931 us), with three of four ignored a quarter of the time. ``cutce_forward`` and
    ``cutce_backward`` take the option as given.

    ``head_layout="vd"``: lm_head_kernel is ``[V, d]`` (a checkpoint's ``[out, in]`` layout, which the
    reference transposes once at load, src/causal_trainer/checkpointing/huggingface.py:1-6). The
    kernels read ``[d, V]`` with the vocabulary contiguous, so this layout costs a transposing copy
    of the head per call (2 B read + 2 B written per element); its gradient comes back as ``[V, d]``, a view
    of the kernels' ``[d, V]``.
    """

    if mesh is None and head_layout in ("dv", "vd") and type(local_chunk_size) is int and local_chunk_size >= 0:
        out = _cut(hidden_states, lm_head_kernel, targets, weights, lm_head_trainable, logits_cache, local_chunk_size,
                   head_layout)
        if out is not None:
            return out
    if head_layout not in ("dv", "vd"):
        raise ValueError("head_layout must be 'dv' ([hidden, vocab]) or 'vd' ([vocab, hidden])")
    if head_layout == "vd":
        if lm_head_kernel.ndim != 2:
            raise ValueError("lm_head_kernel must have shape [vocab, hidden]")
        lm_head_kernel = lm_head_kernel.t()   # (a head that is not dense: made contiguous below)

    local_chunk_size = _integer(local_chunk_size, "local_chunk_size must be a static non-negative integer")
    if local_chunk_size < 0:
        raise ValueError("local_chunk_size must be non-negative")
    layout_ok = hidden_states.ndim == 3
    if not layout_ok:
        raise ValueError("Cut cross-entropy expects hidden_states [batch, sequence, hidden]")
    batch, sequence, hidden = hidden_states.shape
    if tuple(lm_head_kernel.shape[:1]) != (hidden,) or lm_head_kernel.ndim != 2:
        raise ValueError("lm_head_kernel must have shape [hidden, vocab]")
    targets = torch.as_tensor(targets, device=hidden_states.device).to(torch.int32)
    weights = torch.as_tensor(weights, device=hidden_states.device).to(torch.float32)
    for broken, error in (
        (not (targets.shape == weights.shape == (batch, sequence)),
         ValueError("targets and weights must match hidden_states.shape[:-1]")),
        (batch * sequence == 0, ValueError("Cut cross-entropy requires at least one token row")),
        (hidden == 0 or hidden % _HIDDEN_ALIGN != 0,
         ValueError("Cut cross-entropy hidden size must be divisible by 128")),
        (lm_head_kernel.shape[1] == 0, ValueError("Cut cross-entropy requires a non-empty vocabulary")),
        (lm_head_kernel.dtype != hidden_states.dtype,
         TypeError("hidden_states and lm_head_kernel must use the same compute dtype")),
        (not hidden_states.dtype.is_floating_point, TypeError("Cut cross-entropy inputs must have a floating dtype")),
        (hidden_states.dtype != torch.bfloat16,
         TypeError("this build computes Cut cross-entropy in bfloat16 only")),
        (not hidden_states.is_cuda, RuntimeError("Cut cross-entropy is available only on a ROCm GPU")),
    ):
        if broken:
            raise error
    active = _Axes(mesh).beyond_one_device()
    sharded_rows = [axis for axis in ("fsdp", "ep") if axis in active]
    if sharded_rows:
        raise ValueError("Cut cross-entropy currently requires fsdp=ep=1; active unsupported axes: "
                         + ", ".join(sharded_rows))
    if active:
        raise ValueError(f"this build runs on one GPU; mesh axes larger than 1: {active}")
    out = _cut(hidden_states.contiguous(), lm_head_kernel.contiguous(), targets.contiguous(), weights.contiguous(),
               lm_head_trainable, logits_cache, local_chunk_size, "dv")
    if out is None:
        raise RuntimeError("Cut cross-entropy is available only for dense tensors on one ROCm GPU")
    return out


__all__ = ["LOGITS_CACHE_LIMIT_BYTES", "backward_workspace_bytes", "cutce_backward", "cutce_forward", "logits_cache_bytes",
           "pallas_cut_linear_cross_entropy"]
