"""Device-side mirrors of the decoder-layer operations on either side of attention.

``make_position_ids`` / ``rotary_cos_sin`` / ``apply_rotary_cos_sin`` /
``apply_rotary_embedding`` (src/causal_trainer/modeling/rotary.py:63-234) and ``rms_norm``
(src/causal_trainer/modeling/architecture.py:155-162) keep the reference's names, argument
meaning and validation errors; tensors are torch tensors on a ROCm device, bf16 where the
reference's compute dtype is bf16, and the work is done by libct_hotpath.so. ``rms_norm`` and
``apply_rotary_cos_sin`` are differentiable (their backward passes are library kernels too).
"""

from __future__ import annotations

import torch

from . import _lib
from .prep import _dense, _int32, _mask_and_labels, _plain

_STYLES = {"gpt-j": 0, "gpt-neox": 1}


def make_position_ids(attention_mask, segment_ids=None) -> torch.Tensor:
    """Zero-based positions that reset at every packed segment (int32 ``[batch, sequence]``)."""

    plain = _plain("segment_positions", attention_mask, segment_ids)
    if plain is not None:
        return plain
    mask = torch.as_tensor(attention_mask)
    if mask.ndim != 2:
        raise ValueError(f"attention_mask must have shape [batch, sequence], got {tuple(mask.shape)}")
    valid, labels = _mask_and_labels(mask, segment_ids)
    if valid.numel() == 0:
        return torch.empty_like(valid)
    return _dense(_lib.native().segment_positions(valid, labels), "attention_mask and segment_ids")


def rotary_cos_sin(position_ids, inv_freq, dtype=torch.bfloat16):
    """Per-token cos / sin tables ``[batch, sequence, rotary_dim / 2]`` (f32 angles, one cast)."""

    plain = _plain("rotary_tables", position_ids, inv_freq) if dtype == torch.bfloat16 else None
    if plain is not None:
        return plain
    positions = torch.as_tensor(position_ids)
    if positions.ndim != 2:
        raise ValueError(f"position_ids must have shape [batch, sequence], got {tuple(positions.shape)}")
    frequencies = torch.as_tensor(inv_freq)
    if frequencies.ndim != 1 or frequencies.shape[0] == 0:
        raise ValueError(f"inv_freq must be a non-empty vector, got {tuple(frequencies.shape)}")
    if dtype != torch.bfloat16:
        raise ValueError("the MI355X path computes rotary tables in bfloat16 only")
    positions = _int32(positions, "position_ids")
    frequencies = frequencies.to(device=positions.device, dtype=torch.float32).contiguous()
    batch, sequence = positions.shape
    if batch * sequence == 0:
        shape = (batch, sequence, frequencies.shape[0])
        return (torch.empty(shape, dtype=torch.bfloat16, device=positions.device),
                torch.empty(shape, dtype=torch.bfloat16, device=positions.device))
    return _dense(_lib.native().rotary_tables(positions, frequencies), "position_ids and inv_freq")


def apply_rotary_cos_sin(query, key, cosine, sine, *, rope_style: str = "gpt-j", q_scale: float = 1.0):
    """Partial RoPE of Q and K ``[batch, sequence, heads, head_dim]`` from precomputed tables.

    ``q_scale`` (not in the reference signature, default off) also applies the attention
    operator's bf16 pre-scale of Q in the same pass; call the attention operator with scale 1 then.
    """

    if rope_style in _STYLES and type(q_scale) in (float, int):
        try:
            rotated = _lib.native().apply_rotary(query, key, cosine, sine, _STYLES[rope_style], q_scale)
        except TypeError:
            rotated = None      # (something is wrong with the arguments: the validation says what)
        if rotated is not None:
            return rotated
    if query.ndim != 4 or key.ndim != 4:
        raise ValueError("query and key must have shape [batch, sequence, heads, head_dim]")
    if query.shape[:2] != key.shape[:2] or query.shape[-1] != key.shape[-1]:
        raise ValueError(f"incompatible query/key shapes: {tuple(query.shape)} and {tuple(key.shape)}")
    cosine, sine = torch.as_tensor(cosine), torch.as_tensor(sine)
    if cosine.shape != sine.shape:
        raise ValueError(f"cosine and sine shapes differ: {tuple(cosine.shape)} and {tuple(sine.shape)}")
    if cosine.ndim != 3 or cosine.shape[:2] != query.shape[:2]:
        raise ValueError("cosine and sine must have shape "
                         f"[{query.shape[0]}, {query.shape[1]}, rotary_dim / 2], got {tuple(cosine.shape)}")
    rotary_dim = cosine.shape[-1] * 2
    if rotary_dim <= 0 or rotary_dim > query.shape[-1] or rotary_dim % 2:
        raise ValueError(f"invalid rotary dimension {rotary_dim} for head_dim={query.shape[-1]}")
    if rope_style not in _STYLES:
        raise ValueError("rope_style must be 'gpt-j' or 'gpt-neox'")
    if not query.is_cuda:
        raise RuntimeError("query must live on a ROCm GPU")
    if query.dtype != torch.bfloat16 or key.dtype != torch.bfloat16:
        raise ValueError("the MI355X path rotates bfloat16 query and key only")
    cosine = cosine.to(torch.bfloat16).contiguous()
    sine = sine.to(torch.bfloat16).contiguous()
    if query.numel() == 0 or key.numel() == 0:
        raise _lib.CtError(_lib.CT_INVALID_ARGUMENT, "ct_apply_rotary: dimensions must be positive")
    rotated = _lib.native().apply_rotary(query.contiguous(), key.contiguous(), cosine, sine, _STYLES[rope_style],
                                         float(q_scale))
    if rotated is None:
        raise RuntimeError("query, key and the tables must be dense tensors on one ROCm GPU")
    return rotated


def apply_rotary_embedding(query, key, position_ids, inv_freq, *, rope_style: str = "gpt-j"):
    """Partial RoPE of Q and K from positions and inverse frequencies."""

    cosine, sine = rotary_cos_sin(position_ids, inv_freq, query.dtype)
    return apply_rotary_cos_sin(query, key, cosine, sine, rope_style=rope_style)


def rms_norm(x, scale, eps: float, compute_dtype=torch.bfloat16) -> torch.Tensor:
    """RMS normalisation over the last axis with f32 statistics and a learned scale."""

    if compute_dtype == torch.bfloat16:
        try:
            y = _lib.native().rms_norm(x, scale, eps)
        except TypeError:
            y = None    # (something is wrong with the arguments: the validation says what)
        if y is not None:
            return y
    if compute_dtype != torch.bfloat16 or x.dtype != torch.bfloat16:
        raise ValueError("the MI355X path normalises bfloat16 activations with a bfloat16 compute dtype")
    if not x.is_cuda:
        raise RuntimeError("x must live on a ROCm GPU")
    if scale.ndim != 1 or scale.shape[0] != x.shape[-1]:
        raise ValueError(f"scale must have shape ({x.shape[-1]},), got {tuple(scale.shape)}")
    if x.numel() == 0:
        return torch.empty_like(x)
    y = _lib.native().rms_norm(x.contiguous(), scale.to(device=x.device, dtype=torch.bfloat16).contiguous(), float(eps))
    if y is None:
        raise RuntimeError("x and scale must be dense tensors on one ROCm GPU")
    return y


__all__ = ["make_position_ids", "rotary_cos_sin", "apply_rotary_cos_sin", "apply_rotary_embedding", "rms_norm"]
