"""The operators' residuals go through torch's saved-tensor mechanism: hooks (offloading, checkpointing) see each of
them, and the gradients from what the hooks give back are bit for bit those without hooks. What Cut cross-entropy keeps
besides under ``logits_cache=True`` (logits, or an aligned copy of the head) is no residual; without it there is nothing."""

import pytest
import torch
from torch.utils.checkpoint import checkpoint

pytestmark = pytest.mark.gpu


def _operator(ct, gpu, name):
    """(function of the inputs, inputs, gradients of the outputs, (dtype, shape) of every residual)"""

    generator = torch.Generator(device=gpu).manual_seed(17)

    def normal(*shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=generator, device=gpu, dtype=dtype)

    batch, seq, hidden, vocab = 2, 256, 256, 515
    q, k, v = normal(batch, seq, 4, 64), normal(batch, seq, 2, 64), normal(batch, seq, 2, 64)
    targets = torch.randint(vocab, (batch, seq), generator=generator, device=gpu, dtype=torch.int32)
    weights = torch.rand((batch, seq), generator=generator, device=gpu)
    if name == "attention":
        profile = ct.resolve_attention_profile(q.shape, k.shape, None)
        ids = torch.ones((batch, seq), dtype=torch.int32, device=gpu)
        metadata = ct.prepare_attention_metadata(ids, mesh=None, profile=profile)
        inputs, residuals = (q, k, v), [q, k, v, q, normal(batch, seq, 4, dtype=torch.float32)]   # ..., O, LSE
        function = lambda *x: ct.efficient_attention(*x, metadata, profile=profile)  # noqa: E731
    elif name == "rms_norm":
        inputs = residuals = normal(batch, seq, hidden), normal(hidden)
        function = lambda x, scale: ct.rms_norm(x, scale, 1e-6)  # noqa: E731
    elif name == "rotary":
        positions = torch.arange(seq, dtype=torch.int32, device=gpu).repeat(batch, 1)
        tables = ct.rotary_cos_sin(positions, 1e4 ** (-torch.arange(0, 64, 2, device=gpu) / 64))
        inputs, residuals = (q, k), tables
        function = lambda *x: ct.apply_rotary_cos_sin(*x, *tables)  # noqa: E731
    elif name == "sparse_ce":
        inputs = (normal(batch, seq, vocab),)
        residuals = [*inputs, targets, weights, weights]      # ..., LSE
        function = lambda x: ct.pallas_fused_sparse_cross_entropy(x, targets, weights)  # noqa: E731
    else:
        inputs = normal(batch, seq, hidden), normal(hidden, vocab)
        residuals = [*inputs, targets, weights, weights.view(-1)]
        function = lambda x, w: ct.pallas_cut_linear_cross_entropy(x, w, targets, weights)[0]  # noqa: E731
    inputs = tuple(t.requires_grad_(True) for t in inputs)
    with torch.no_grad():
        outputs = function(*inputs)
    outputs = outputs if isinstance(outputs, tuple) else (outputs,)
    cotangents = tuple(normal(*t.shape, dtype=t.dtype) for t in outputs)
    return function, inputs, cotangents, sorted((str(t.dtype), tuple(t.shape)) for t in residuals)


@pytest.mark.parametrize("name", ["attention", "rms_norm", "rotary", "sparse_ce", "cut_ce"])
def test_residuals_pass_the_saved_tensor_hooks(ct, gpu, name):
    function, inputs, cotangents, residuals = _operator(ct, gpu, name)

    def gradients(call):
        outputs = call()
        return torch.autograd.grad(outputs, inputs, cotangents if isinstance(outputs, tuple) else cotangents[0])

    expected = gradients(lambda: function(*inputs))
    packed = []

    def pack(tensor):
        packed.append((str(tensor.dtype), tuple(tensor.shape)))
        return tensor.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda tensor: tensor.to(gpu)):
        offloaded = gradients(lambda: function(*inputs))
    assert sorted(packed) == residuals
    recomputed = gradients(lambda: checkpoint(function, *inputs, use_reentrant=False))
    for other in (offloaded, recomputed):
        assert all(torch.equal(a, b) for a, b in zip(expected, other))


@pytest.mark.parametrize("vocab,layout", [(512, "dv"), (515, "dv"), (515, "vd")])
def test_cut_ce_without_a_logits_cache_keeps_its_residuals_only(ct, gpu, vocab, layout):
    """Device memory held between the two directions, with an aligned head and with one that the kernels copy: the
    outputs and ``lse`` (of a [V, d] head also the transposed copy, which is its residual), and under hooks that
    offload every residual the outputs alone."""

    rows, hidden = 512, 256
    generator = torch.Generator(device=gpu).manual_seed(3)
    normal = lambda *shape: torch.randn(shape, generator=generator, device=gpu, dtype=torch.bfloat16)  # noqa: E731
    x = normal(1, rows, hidden).requires_grad_(True)
    head = (normal(hidden, vocab) if layout == "dv" else normal(vocab, hidden)).requires_grad_(True)
    targets = torch.randint(vocab, (1, rows), generator=generator, device=gpu, dtype=torch.int32)
    weights = torch.ones((1, rows), device=gpu)

    def kept():
        before = torch.cuda.memory_allocated()
        outputs = ct.pallas_cut_linear_cross_entropy(x, head, targets, weights, logits_cache=False, head_layout=layout)
        held = torch.cuda.memory_allocated() - before
        torch.autograd.grad(outputs[0], (x, head))
        return held

    kept()                                  # (what a first call sets up for good)
    outputs = 2 * 512                       # two scalars, in the allocator's units of 512 bytes
    transposed = 2 * hidden * 768 if layout == "vd" else 0      # rows padded to a multiple of 256
    assert kept() == outputs + 4 * rows + transposed
    with torch.autograd.graph.saved_tensors_hooks(lambda tensor: tensor.cpu(), lambda tensor: tensor.to(gpu)):
        assert kept() == outputs
