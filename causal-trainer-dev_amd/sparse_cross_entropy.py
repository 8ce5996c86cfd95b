"""Sparse cross-entropy on materialised logits, the trainer's non-fused loss backend.

Mirrors ``pallas_fused_sparse_cross_entropy`` (src/causal_trainer/kernels/cross_entropy.py:600-643;
per-token f32 losses, custom VJP with the analytic logits gradient, rows with target -100 or
weight 0 contribute nothing and are not read) on one MI355X: same name, argument meaning and
shape errors; ``mesh`` is accepted for signature compatibility and must describe one device.
"""

from __future__ import annotations

import torch

from . import _lib

_DTYPES = (torch.bfloat16, torch.float32)


def pallas_fused_sparse_cross_entropy(logits, targets, weights, *, mesh=None) -> torch.Tensor:
    """Per-token weighted CE ``[batch, sequence]`` (f32) of logits ``[batch, sequence, vocab]``."""

    if mesh is None:
        try:
            loss = _lib.native().sparse_ce(logits, targets, weights)
        except TypeError:
            loss = None     # (something is wrong with the arguments: the validation says what)
        if loss is not None:
            return loss
    if logits.ndim != 3 or tuple(targets.shape) != tuple(logits.shape[:-1]) or tuple(weights.shape) != tuple(targets.shape):
        raise ValueError("Pallas CE expects logits [batch, sequence, vocab] and matching target/weight rows")
    if mesh is not None and getattr(mesh, "size", 1) != 1:
        raise ValueError("this build runs on one device: pass mesh=None or a one-device mesh")
    if not logits.is_cuda:
        raise RuntimeError("logits must live on a ROCm GPU")
    if logits.dtype not in _DTYPES:
        raise ValueError("logits must be bfloat16 or float32")
    leading = logits.shape[:-1]
    if logits.numel() == 0:
        return torch.zeros(leading, dtype=torch.float32, device=logits.device)
    loss = _lib.native().sparse_ce(
        logits.contiguous(), targets.to(device=logits.device, dtype=torch.int32).contiguous(),
        weights.to(device=logits.device, dtype=torch.float32).contiguous())
    if loss is None:
        raise RuntimeError("logits must be a dense tensor on a ROCm GPU")
    return loss


__all__ = ["pallas_fused_sparse_cross_entropy"]
