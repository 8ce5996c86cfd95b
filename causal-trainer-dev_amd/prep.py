"""Device-side mirrors of the two preparation functions directly in front of the hot paths.

``canonicalize_segment_ids`` (src/causal_trainer/modeling/rotary.py:13-50) and
``shifted_targets_and_weights`` (``_shifted_targets_and_weights``,
src/causal_trainer/training/losses.py:21-85) keep the reference's argument meaning and
validation errors; tensors are torch tensors on a ROCm device and the work is done by
libct_hotpath.so. They define which tokens attention may connect and which rows the loss
ignores, so they are integer kernels that match the reference bit for bit.
"""

from __future__ import annotations

import torch

from . import _lib


def _int32(tensor, name: str, shape=None) -> torch.Tensor:
    tensor = torch.as_tensor(tensor)
    if not tensor.is_cuda:
        raise RuntimeError(f"{name} must live on a ROCm GPU")
    if shape is not None and tuple(tensor.shape) != tuple(shape):
        raise ValueError(f"{name} must have shape {tuple(shape)}, got {tuple(tensor.shape)}")
    return tensor.contiguous() if tensor.dtype == torch.int32 else tensor.to(torch.int32).contiguous()


def _nonzero(tensor, name: str) -> torch.Tensor:
    """A mask for the kernels that read "not zero" as set: int32 as it is, anything else compared first."""

    tensor = torch.as_tensor(tensor)
    return _int32(tensor if tensor.dtype == torch.int32 else tensor != 0, name)


def _dense(result, names: str):
    """What the native side returned, an error if it did not take the arguments."""

    if result is None:
        raise RuntimeError(f"{names} must be dense tensors on one ROCm GPU, without forward-mode tangents")
    return result


def _plain(name: str, *arguments):
    """The native function on arguments as they come, None where it does not take them: the validation then says why
    or normalises them. A third of a call's host time is that validation (canonical ids 6.8 -> 4.8 us, targets 9.3 -> 5.9)."""

    try:
        return getattr(_lib.native(), name)(*arguments)
    except TypeError:
        return None


def _mask_and_labels(mask, segment_ids):
    valid = _nonzero(mask, "attention_mask")
    if segment_ids is None:
        return valid, None
    labels = torch.as_tensor(segment_ids)
    if labels.shape != valid.shape:
        raise ValueError(f"segment_ids must have shape {tuple(valid.shape)}, got {tuple(labels.shape)}")
    return valid, _int32(labels, "segment_ids")


def canonicalize_segment_ids(attention_mask, segment_ids=None) -> torch.Tensor:
    """One-based ids of contiguous valid runs, zero for padding (int32 ``[batch, sequence]``)."""

    plain = _plain("canonical_ids", attention_mask, segment_ids)
    if plain is not None:
        return plain
    mask = torch.as_tensor(attention_mask)
    if mask.ndim != 2:
        raise ValueError(f"attention_mask must have shape [batch, sequence], got {tuple(mask.shape)}")
    valid, labels = _mask_and_labels(mask, segment_ids)
    if valid.numel() == 0:
        return torch.empty_like(valid)
    return _dense(_lib.native().canonical_ids(valid, labels), "attention_mask and segment_ids")


def shifted_targets_and_weights(input_ids, attention_mask, segment_ids=None, assistant_mask=None,
                                loss_mask=None, labels=None, *, ignore_index: int = -100):
    """Safe shifted targets (int32) and target-position loss weights (f32), both ``[batch, sequence - 1]``."""

    plain = _plain("shifted_targets", input_ids, attention_mask, segment_ids, assistant_mask, loss_mask, labels, ignore_index)
    if plain is not None:
        return plain
    tokens = torch.as_tensor(input_ids)
    if tokens.ndim != 2:
        raise ValueError(f"input_ids must have shape [batch, sequence], got {tuple(tokens.shape)}")
    tokens = _int32(tokens, "input_ids")
    shape = tokens.shape
    label_t = None if labels is None else _int32(labels, "labels", shape)
    # validity is "mask == 1": other values, True included as 1, follow the reference's comparison
    mask_t = None if attention_mask is None else _int32(attention_mask, "attention_mask", shape)
    segment_t = None if segment_ids is None else _int32(segment_ids, "segment_ids", shape)
    assistant_t = None
    if assistant_mask is not None:
        assistant = torch.as_tensor(assistant_mask)
        if tuple(assistant.shape) != tuple(shape):
            raise ValueError(f"assistant_mask must have shape {tuple(shape)}, got {tuple(assistant.shape)}")
        assistant_t = _nonzero(assistant, "assistant_mask")
    loss_t = None
    if loss_mask is not None:
        loss_t = torch.as_tensor(loss_mask)
        if tuple(loss_t.shape) != tuple(shape):
            raise ValueError(f"loss_mask must have shape {tuple(shape)}, got {tuple(loss_t.shape)}")
        loss_t = loss_t.to(torch.float32).contiguous()
    batch, sequence = shape
    if sequence < 2:
        raise ValueError("input_ids needs at least two positions to form a prediction edge")
    if batch == 0:
        raise _lib.CtError(_lib.CT_INVALID_ARGUMENT, "ct_shifted_targets_and_weights: batch and sequence must be positive, "
                           f"got [{batch}, {sequence}]")
    return _dense(_lib.native().shifted_targets(tokens, mask_t, segment_t, assistant_t, loss_t, label_t, int(ignore_index)),
                  "input_ids and the masks")


__all__ = ["canonicalize_segment_ids", "shifted_targets_and_weights"]
