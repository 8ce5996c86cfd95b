"""CPU-only checks of the host-side mirror and of the C ABI surface (no compute calls)."""

import ctypes
import importlib.util
import re
import sys
import threading
import time
from pathlib import Path

import numpy as np
import pytest
import torch

ROOT = Path(__file__).resolve().parents[1]


def test_library_exports_every_declared_symbol(ct):
    header = (ROOT / "include" / "ct_hotpath.h").read_text()
    declared = set(re.findall(r"\b(ct_[a-z0-9_]+)\s*\(", header))
    assert declared == set(ct._lib.SYMBOLS), declared ^ set(ct._lib.SYMBOLS)
    library = ct._lib.load()
    for name in declared:
        assert hasattr(library, name), name
    assert library.ct_abi_version() == ct._lib.ABI_VERSION
    assert library.ct_last_error() == b"" or isinstance(library.ct_last_error(), bytes)


def test_size_queries_need_no_gpu(ct):
    library = ct._lib.load()
    nrb = 4096 // 32
    bins = sum(33 + 4 * ((nrb + pb - 1) // pb) for pb in (2, 4, 8))
    assert library.ct_attn_meta_bytes(4, 4096) == (4 * (nrb * 12 + 2 * nrb + nrb // 4) + bins) * 4
    assert library.ct_attn_meta_bytes(0, 128) == 0
    # the backward's scratch: the work list, statistics and partial sums alone are small ...
    least = library.ct_attn_bwd_workspace_bytes(4, 4096, 32, 8, 128)
    assert 0 < least < 1 << 30
    assert library.ct_attn_bwd_workspace_bytes(4, 4000, 32, 8, 128) == 0
    assert library.ct_attn_bwd_workspace_bytes_from_ds(4, 4000, 32, 8, 128, 0) == 0
    # ... the stored-dS form adds 2 KB per (key block, query block at or after it) pair of every
    # batch row and query head (nrb^2 pairs with visible ends)
    causal = library.ct_attn_bwd_workspace_bytes_from_ds(4, 4096, 32, 8, 128, 0)
    hybrid = library.ct_attn_bwd_workspace_bytes_from_ds(4, 4096, 32, 8, 128, 1)
    assert causal - least == 4 * 32 * (nrb * (nrb + 1) // 2) * 2048
    assert hybrid - least == 4 * 32 * nrb * nrb * 2048
    # the region is capped at 16 GiB but never below one KV head's blocks: 64 query heads over 8 KV heads
    # at S = 32768 take 8.6 GB per KV head, so the backward runs in 8 passes of one KV head
    long_blocks = (32768 // 32) * (32768 // 32 + 1) // 2
    long_total = library.ct_attn_bwd_workspace_bytes_from_ds(1, 32768, 64, 8, 128, 0)
    long_least = library.ct_attn_bwd_workspace_bytes(1, 32768, 64, 8, 128)
    assert 8 * long_blocks * 2048 <= long_total - long_least + (1 << 30) and long_total < 10 << 30
    # one KV head beyond 64 GiB: that form is not available
    assert library.ct_attn_bwd_workspace_bytes_from_ds(1, 1 << 20, 2, 1, 64, 1) == 0
    shape = ct._lib.CutceShape(16384, 4096, 128256)
    fwd = library.ct_cutce_fwd_workspace_bytes(ctypes.byref(shape))
    full = library.ct_cutce_bwd_workspace_bytes(ctypes.byref(shape))
    least = library.ct_cutce_bwd_workspace_min_bytes(ctypes.byref(shape))
    assert 0 < fwd < 64 << 20
    assert full >= 16384 * 128256 * 2
    assert 0 < least < full


def test_argument_validation_happens_before_any_launch(ct):
    library = ct._lib.load()
    args = ct._lib.AttnFwdArgs(batch=1, seq=100, q_heads=4, kv_heads=2, head_dim=128, scale=0.1)
    assert library.ct_attn_fwd(None, ctypes.byref(args)) == ct._lib.CT_INVALID_ARGUMENT
    assert b"null pointer" in library.ct_last_error()
    for field in ("q", "k", "v", "segment_ids", "tile_meta", "out", "lse"):
        setattr(args, field, 4096)       # never dereferenced: validation fails first
    assert library.ct_attn_fwd(None, ctypes.byref(args)) == ct._lib.CT_INVALID_ARGUMENT
    assert b"128-aligned" in library.ct_last_error()
    args.seq, args.q_heads, args.kv_heads = 128, 5, 2
    assert library.ct_attn_fwd(None, ctypes.byref(args)) == ct._lib.CT_INVALID_ARGUMENT
    assert b"divisible by the KV head count" in library.ct_last_error()
    args.q_heads, args.head_dim = 4, 96
    assert library.ct_attn_fwd(None, ctypes.byref(args)) == ct._lib.CT_UNSUPPORTED
    args.head_dim, args.k = 128, 4096 + 8
    assert library.ct_attn_fwd(None, ctypes.byref(args)) == ct._lib.CT_INVALID_ARGUMENT
    assert b"16-byte aligned" in library.ct_last_error()
    shape = ct._lib.CutceShape(10, 100, 50)
    cargs = ct._lib.CutceFwdArgs(shape=shape)
    for field in ("hidden", "head", "targets", "weights", "nll_sum", "weight_sum", "lse", "workspace"):
        setattr(cargs, field, 4096)
    assert library.ct_cutce_fwd(None, ctypes.byref(cargs)) == ct._lib.CT_INVALID_ARGUMENT
    assert b"divisible by 128" in library.ct_last_error()
    cargs.shape = ct._lib.CutceShape(10, 128, 50)
    cargs.workspace_bytes = 16
    assert library.ct_cutce_fwd(None, ctypes.byref(cargs)) == ct._lib.CT_WORKSPACE_TOO_SMALL


def test_cutce_backward_refuses_strides_beyond_its_32_bit_offsets(ct):
    """Tiles of 256 rows, 2 bytes an element: a stride of 2^23 is the last whose offsets stay below 4 GiB. In reach,
    the call gets as far as its workspace."""

    library = ct._lib.load()
    args = ct._lib.CutceBwdArgs(workspace_bytes=16)
    for field in ("hidden", "head", "targets", "weights", "lse", "dy", "dhidden", "workspace"):
        setattr(args, field, 4096)       # never dereferenced: validation fails first
    for rows, vocab, dhead, status in (
            (10, 1 << 23, 4096, ct._lib.CT_WORKSPACE_TOO_SMALL), (10, (1 << 23) + 1, 4096, ct._lib.CT_UNSUPPORTED),
            (10, (1 << 23) + 1, None, ct._lib.CT_UNSUPPORTED), (1 << 23, 50, 4096, ct._lib.CT_WORKSPACE_TOO_SMALL),
            ((1 << 23) + 1, 50, 4096, ct._lib.CT_UNSUPPORTED), ((1 << 23) + 1, 50, None, ct._lib.CT_WORKSPACE_TOO_SMALL)):
        args.shape, args.dhead = ct._lib.CutceShape(rows, 128, vocab), dhead
        assert library.ct_cutce_bwd(None, ctypes.byref(args)) == status, (rows, vocab, dhead, library.ct_last_error())


def test_cutce_panel_and_logits_cache_cannot_be_mixed_up(ct):
    """A forward with a lent panel writes no panel into its logits cache: the cache it takes is one that the backward
    without a panel refuses, and the other way round. A panel that is too short is refused too. (No workspace or a
    misaligned output ends the calls that get past these checks, so nothing is launched.)"""

    library, shape = ct._lib.load(), ct._lib.CutceShape(10, 128, 1031)
    query = lambda name: int(getattr(library, name)(ctypes.byref(shape)))  # noqa: E731
    panel, with_panel = query("ct_cutce_panel_bytes"), query("ct_cutce_logits_cache_bytes")
    assert panel == 128 * 1280 * 2 and with_panel == 256 * 1280 * 4 + panel
    forward = ct._lib.CutceFwdArgs(shape=shape, logits_cache=4096, workspace_bytes=query("ct_cutce_fwd_workspace_bytes"))
    for field in ("hidden", "head", "targets", "weights", "nll_sum", "weight_sum", "lse", "workspace"):
        setattr(forward, field, 4096)       # never dereferenced: validation fails first
    backward = ct._lib.CutceBwdArgs(shape=shape, logits_cache=4096, workspace_bytes=16)
    for field in ("hidden", "head", "targets", "weights", "lse", "dy", "dhidden", "workspace"):
        setattr(backward, field, 4096)
    refused, short, misaligned = ct._lib.CT_INVALID_ARGUMENT, ct._lib.CT_WORKSPACE_TOO_SMALL, 4096 + 2

    def run(cache_bytes, lent, lent_bytes):
        forward.logits_cache_bytes = backward.logits_cache_bytes = cache_bytes
        return (library.ct_cutce_fwd_panel(None, ctypes.byref(forward), lent, lent_bytes, 1),
                library.ct_cutce_bwd_panel(None, ctypes.byref(backward), lent, lent_bytes))

    for cache_bytes in (with_panel, with_panel - panel + 16, 2 * with_panel):
        assert run(cache_bytes, 4096, panel) == (refused, refused)
        assert b"without room for one" in library.ct_last_error()
    assert run(with_panel - panel - 16, 4096, panel) == (short, short)
    assert run(with_panel - panel, 4096, panel - 2) == (short, short)
    assert b"panel" in library.ct_last_error()
    assert run(with_panel - panel, misaligned, panel) == (refused, refused)
    assert run(with_panel - panel, None, 0) == (short, short)         # what a forward with a panel has filled
    assert b"logits cache" in library.ct_last_error()
    assert library.ct_cutce_bwd(None, ctypes.byref(backward)) == short and b"logits cache" in library.ct_last_error()
    # the sizes that belong together pass these checks: the backward gets as far as its workspace
    for cache_bytes, lent, lent_bytes in ((with_panel - panel, 4096, panel), (with_panel, None, 0)):
        backward.logits_cache_bytes = cache_bytes
        assert library.ct_cutce_bwd_panel(None, ctypes.byref(backward), lent, lent_bytes) == short
        assert b"workspace" in library.ct_last_error()


@pytest.mark.parametrize("rows,hidden,vocab,both", [
    (512, 512, 150001, 1), (513, 512, 150001, 0),       # many rows and a large head: one copy for both directions is faster
    (640, 768, 100003, 0), (1000, 1024, 32003, 1),      # ... up to 35 million elements it is not
    (1024, 2048, 16001, 1), (1024, 2048, 17091, 0),
    (1025, 1024, 16001, 0), (64, 1024, 16000, 0),       # too many rows for the backward; a head that is aligned
])
def test_cutce_heads_that_both_directions_read_in_place(ct, rows, hidden, vocab, both):
    shape = ct._lib.CutceShape(rows, hidden, vocab)
    assert ct._lib.load().ct_cutce_head_in_place(ctypes.byref(shape)) == both


@pytest.mark.parametrize("rows,hidden,vocab,forward,backward,both", [
    (64, 4096, 150001, True, True, True), (768, 1024, 50257, True, True, False), (769, 1024, 50257, True, False, False),
    (700, 512, 5001, False, False, False), (64, 1024, 16000, False, False, False)])
def test_cutce_sizes_leave_out_a_copy_that_nobody_makes(ct, rows, hidden, vocab, forward, backward, both):
    """A direction that reads the head in place uses the copy of 256 columns; whoever lends a panel still finds its bytes
    in the sizes that the panel's are to be taken from."""

    library, shape = ct._lib.load(), ct._lib.CutceShape(rows, hidden, vocab)
    query = lambda name: int(getattr(library, name)(ctypes.byref(shape)))  # noqa: E731
    panel, tail = query("ct_cutce_panel_bytes"), hidden * 256 * 2
    least = query("ct_cutce_fwd_workspace_min_bytes")
    logits = (rows + 255) // 256 * 256 * ((vocab + 255) // 256 * 256) * 4
    assert query("ct_cutce_fwd_workspace_bytes") - least == panel and query("ct_cutce_logits_cache_bytes") - logits == panel
    assert query("ct_cutce_fwd_workspace_used_bytes") - least == (tail if forward else panel)
    assert query("ct_cutce_logits_cache_used_bytes") - logits == (tail if both else panel)
    spared = query("ct_cutce_bwd_workspace_bytes") - query("ct_cutce_bwd_workspace_used_bytes")
    assert spared == (panel - tail if backward else 0) and query("ct_cutce_bwd_workspace_bytes") > panel
    # what the operators allocate
    assert ct.cut_cross_entropy.logits_cache_bytes(rows, hidden, vocab) == query("ct_cutce_logits_cache_used_bytes")
    assert ct.cut_cross_entropy.backward_workspace_bytes(rows, hidden, vocab) == query("ct_cutce_bwd_workspace_used_bytes")
    bounded = ct.cut_cross_entropy.backward_workspace_bytes(rows, hidden, vocab, 16)
    floor, share = query("ct_cutce_bwd_workspace_min_bytes"), query("ct_cutce_bwd_workspace_bytes")
    # (a bound is the share of the whole that it has always been, and no more than is used)
    assert bounded == min(floor + (share - floor) * 16 // rows, query("ct_cutce_bwd_workspace_used_bytes"))


@pytest.mark.parametrize("torch_side", ["absent", "broken", "there"])
def test_library_is_linked_whatever_becomes_of_the_torch_side(monkeypatch, tmp_path, torch_side):
    """libct_hotpath.so needs hipcc only: it is linked without torch, and before a torch side that fails to compile
    (which is still an error)."""

    spec = importlib.util.spec_from_file_location("build_recipe", ROOT / "causal-trainer-dev_amd" / "build.py")
    recipe = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(recipe)
    made = []

    def run(command):
        output = Path(command[command.index("-o") + 1]).name
        if torch_side == "broken" and output == "ct_torch.o":
            raise RuntimeError("no g++")
        made.append(output)

    monkeypatch.setattr(recipe, "PACKAGE_DIR", tmp_path)
    monkeypatch.setattr(recipe, "hipcc", lambda: "hipcc")
    monkeypatch.setattr(recipe, "_run", run)
    monkeypatch.setattr(recipe.importlib.util, "find_spec", lambda name: None if torch_side == "absent" else spec)
    if torch_side == "broken":
        with pytest.raises(RuntimeError, match="no g"):
            recipe.build()
    else:
        assert recipe.build() == recipe.LIBRARY
    objects = {Path(name).stem + ".o" for name in recipe.SOURCES} | ({"ct_torch.o"} if torch_side == "there" else set())
    assert set(made[:len(objects)]) == objects
    assert made[len(objects):] == ["libct_hotpath.so"] + (["_native.so"] if torch_side == "there" else [])


def test_native_operators_let_other_threads_run(ct):
    """The native functions give the GIL up while they work: with Python's own switching as good as off, a waiting
    thread still gets its turn (after a few dozen calls; a call that keeps the GIL never lets it in)."""

    native, x = ct._lib.native(), torch.zeros(2, 128)
    go, ran, interval = threading.Lock(), [], sys.getswitchinterval()
    go.acquire()

    def other():
        go.acquire()
        ran.append(True)

    thread = threading.Thread(target=other)
    thread.start()
    sys.setswitchinterval(1000)
    try:
        go.release()
        deadline = time.monotonic() + 10
        while not ran and time.monotonic() < deadline:
            assert native.rms_norm(x, x, 1e-6) is None     # (not on a GPU: the wrapper's validation would say so)
        assert ran
    finally:
        sys.setswitchinterval(interval)
        thread.join()


def test_profile_resolution_matches_reference_tiers(ct):
    # tests/kernels/test_efficient_attention.py:226-249: S=4096, 32 heads, tp=4 -> h8, q256, kv 512/256
    profile = ct.resolve_attention_profile((4, 4096, 32, 128), (4, 4096, 1, 128), {"tp": 4})
    assert (profile.block_h, profile.block_q, profile.block_kv_outer, profile.block_kv_compute) == (8, 256, 512, 256)
    long_profile = ct.resolve_attention_profile((1, 32768, 64, 128), (1, 32768, 8, 128), None)
    assert (long_profile.block_kv_outer, long_profile.block_kv_compute) == (1024, 256)
    hybrid = ct.resolve_attention_profile((2, 8192, 16, 128), (2, 8192, 16, 128), None, has_attention_end=True)
    assert hybrid.block_h * hybrid.block_q <= 2048 and hybrid.block_q % 128 == 0
    assert ct.default_attention_scale(128) == 128 ** -0.5
    with pytest.raises(ValueError, match="128-aligned"):
        ct.resolve_attention_profile((1, 100, 2, 128), (1, 100, 1, 128), None)
    with pytest.raises(ValueError, match="divisible by the KV head count"):
        ct.resolve_attention_profile((1, 128, 3, 128), (1, 128, 2, 128), None)


def test_attention_argument_errors(ct):
    q = torch.zeros((1, 128, 2, 128), dtype=torch.bfloat16)
    k = torch.zeros((1, 128, 1, 128), dtype=torch.bfloat16)
    meta = ct.AttentionMetadata(*(torch.zeros((1, 128), dtype=torch.int32),) * 2,
                                torch.zeros((1, 1, 2), dtype=torch.int32),
                                torch.zeros((1, 1, 2), dtype=torch.int32))
    # tests/kernels/test_efficient_attention.py:420-441: non-causal is rejected
    with pytest.raises(ValueError, match="implements causal attention only"):
        ct.efficient_attention(q, k, k, meta, causal=False)
    with pytest.raises(TypeError, match="compile-time bool"):
        ct.efficient_attention(q, k, k, meta, causal=1)
    with pytest.raises(TypeError, match="requires BF16"):
        ct.efficient_attention(q.float(), k.float(), k.float(), meta)
    with pytest.raises(ValueError, match="key and value shapes differ"):
        ct.efficient_attention(q, k, k[:, :64], meta)
    with pytest.raises(ValueError, match="head_dim"):
        ct.efficient_attention(q[..., :32], k[..., :32], k[..., :32], meta)
    with pytest.raises(ValueError, match="one GPU"):
        ct.efficient_attention(q, k, k, meta, mesh={"tp": 2})
    with pytest.raises(RuntimeError, match="only on a ROCm GPU"):
        ct.efficient_attention(q, k, k, meta)


def test_cutce_argument_errors(ct):
    fn = ct.pallas_cut_linear_cross_entropy
    hidden = torch.zeros((1, 4, 128), dtype=torch.bfloat16)
    head = torch.zeros((128, 10), dtype=torch.bfloat16)
    targets = torch.zeros((1, 4), dtype=torch.int32)
    weights = torch.ones((1, 4))
    with pytest.raises(ValueError, match=r"\[batch, sequence, hidden\]"):
        fn(hidden[0], head, targets, weights)
    with pytest.raises(ValueError, match=r"\[hidden, vocab\]"):
        fn(hidden, head.T, targets, weights)
    with pytest.raises(ValueError, match="must match hidden_states"):
        fn(hidden, head, targets[:, :2], weights)
    with pytest.raises(ValueError, match="divisible by 128"):
        fn(hidden[..., :100], head[:100], targets, weights)
    with pytest.raises(TypeError, match="same compute dtype"):
        fn(hidden, head.float(), targets, weights)
    with pytest.raises(TypeError, match="non-negative integer"):
        fn(hidden, head, targets, weights, local_chunk_size=True)
    with pytest.raises(ValueError, match="non-negative"):
        fn(hidden, head, targets, weights, local_chunk_size=-1)
    # tests/kernels/test_tiled_cut.py:158-166: every invalid chunk size names the option
    for invalid in (True, 1.5, "128", -1):
        with pytest.raises((TypeError, ValueError), match="local_chunk_size"):
            fn(hidden, head, targets, weights, local_chunk_size=invalid)
    # the head as [vocab, hidden]: named by the option, checked like the other layout
    with pytest.raises(ValueError, match="head_layout"):
        fn(hidden, head, targets, weights, head_layout="vocab_major")
    with pytest.raises(ValueError, match=r"\[hidden, vocab\]"):
        fn(hidden, head, targets, weights, head_layout="vd")
    with pytest.raises(RuntimeError, match="only on a ROCm GPU"):
        fn(hidden, head.T.contiguous(), targets, weights, head_layout="vd")
    with pytest.raises(RuntimeError, match="only on a ROCm GPU"):
        fn(hidden, head, targets, weights)


def test_local_chunk_size_bounds_the_backward_workspace(ct):
    # cut_cross_entropy.py:697-825: the chunk option exists to bound transient memory
    from causal_trainer_dev_amd.cut_cross_entropy import backward_workspace_bytes

    rows, hidden, vocab = 16384, 4096, 128256
    library = ct._lib.load()
    shape = ct._lib.CutceShape(rows, hidden, vocab)
    full = library.ct_cutce_bwd_workspace_bytes(ctypes.byref(shape))
    least = library.ct_cutce_bwd_workspace_min_bytes(ctypes.byref(shape))
    assert backward_workspace_bytes(rows, hidden, vocab, 0) == full
    assert backward_workspace_bytes(rows, hidden, vocab, rows) == full
    sizes = [backward_workspace_bytes(rows, hidden, vocab, chunk) for chunk in (8192, 2048, 512, 1)]
    assert sizes == sorted(sizes, reverse=True) and all(least <= size < full for size in sizes)
    assert sizes[1] < full // 4 and sizes[-1] < least + (1 << 20)
    # the slab part shrinks in proportion to the chunk
    assert abs((sizes[1] - least) - (full - least) // 8) <= 1


def _ffi_handlers_in_source():
    """name -> (operands, results, attribute names) from the XLA_FFI_DEFINE_HANDLER_SYMBOL blocks."""

    source = (ROOT / "causal-trainer-dev_amd" / "csrc" / "ct_ffi.cc").read_text()
    found = {}
    for block in re.findall(r"XLA_FFI_DEFINE_HANDLER_SYMBOL\((.*?)\);\n", source, flags=re.S):
        name = block.split(",", 1)[0].strip()
        attributes = tuple(re.findall(r'\.Attr<[^>]+>\("(\w+)"\)', block))
        found[name] = (len(re.findall(r"\.Arg<", block)), len(re.findall(r"\.Ret<", block)), attributes)
    return found


def test_jax_binding_matches_the_ffi_handlers_and_the_documentation(ct):
    """The JAX side cannot run here (no jax): what can be held is static agreement between the
    handlers csrc/ct_ffi.cc defines, the table and call sites of jax_ffi.py, and the integration document."""

    import ast
    import inspect

    from causal_trainer_dev_amd import jax_ffi

    in_source = _ffi_handlers_in_source()
    assert len(in_source) == 14
    assert {name: tuple(handler) for name, handler in jax_ffi.HANDLERS.items()} == in_source
    documented = set(re.findall(r"`(ct_ffi_\w+)`", (ROOT / "INTEGRATION.md").read_text()))
    assert documented == set(in_source)

    # every _call site names a known handler and passes the operand / result / attribute counts
    tree = ast.parse(inspect.getsource(jax_ffi))
    sites = [node for node in ast.walk(tree)
             if isinstance(node, ast.Call) and getattr(node.func, "id", None) == "_call"]
    assert len(sites) >= 5
    for site in sites:
        name = site.args[0].value
        operands, results, attributes = in_source[name]
        assert isinstance(site.args[1], ast.List) and len(site.args[1].elts) == results, name
        assert len(site.args) - 2 == operands, name
        assert tuple(keyword.arg for keyword in site.keywords) == attributes, name
    # every registered handler has a caller: no symbol is handed to a maintainer without its glue
    used = {site.args[0].value for site in sites}
    assert used == set(in_source)

    # the operators keep the reference's signatures (efficient_attention.py:326-331, :1890-1900;
    # cut_cross_entropy.py:828-838)
    def parameters(function):
        return [(p.name, p.kind.name, p.default) for p in inspect.signature(function).parameters.values()]

    empty = inspect.Parameter.empty
    assert parameters(jax_ffi.efficient_attention) == [
        ("query", "POSITIONAL_OR_KEYWORD", empty), ("key", "POSITIONAL_OR_KEYWORD", empty),
        ("value", "POSITIONAL_OR_KEYWORD", empty), ("metadata", "POSITIONAL_OR_KEYWORD", empty),
        ("mesh", "KEYWORD_ONLY", empty), ("profile", "KEYWORD_ONLY", None), ("scale", "KEYWORD_ONLY", None),
        ("causal", "KEYWORD_ONLY", True)]
    assert parameters(jax_ffi.prepare_attention_metadata) == [
        ("canonical_segment_ids", "POSITIONAL_OR_KEYWORD", empty), ("mesh", "KEYWORD_ONLY", empty),
        ("profile", "KEYWORD_ONLY", empty), ("attention_end", "KEYWORD_ONLY", None)]
    assert parameters(jax_ffi.pallas_cut_linear_cross_entropy) == [
        ("hidden_states", "POSITIONAL_OR_KEYWORD", empty), ("lm_head_kernel", "POSITIONAL_OR_KEYWORD", empty),
        ("targets", "POSITIONAL_OR_KEYWORD", empty), ("weights", "POSITIONAL_OR_KEYWORD", empty),
        ("mesh", "KEYWORD_ONLY", empty), ("sparse_compaction", "KEYWORD_ONLY", False),
        ("lm_head_trainable", "KEYWORD_ONLY", True), ("local_chunk_size", "KEYWORD_ONLY", 0)]
    # the rows either side of the two paths (rotary.py:13-16, :63-66, :132-136, :160-167, :207-214;
    # architecture.py:155; losses.py:21-30; cross_entropy.py:600-606)
    assert parameters(jax_ffi.canonicalize_segment_ids) == [
        ("attention_mask", "POSITIONAL_OR_KEYWORD", empty), ("segment_ids", "POSITIONAL_OR_KEYWORD", None)]
    assert parameters(jax_ffi.make_position_ids) == parameters(jax_ffi.canonicalize_segment_ids)
    assert parameters(jax_ffi.rotary_cos_sin) == [
        ("position_ids", "POSITIONAL_OR_KEYWORD", empty), ("inv_freq", "POSITIONAL_OR_KEYWORD", empty),
        ("dtype", "POSITIONAL_OR_KEYWORD", empty)]
    assert parameters(jax_ffi.apply_rotary_cos_sin)[:5] == [
        ("query", "POSITIONAL_OR_KEYWORD", empty), ("key", "POSITIONAL_OR_KEYWORD", empty),
        ("cosine", "POSITIONAL_OR_KEYWORD", empty), ("sine", "POSITIONAL_OR_KEYWORD", empty),
        ("rope_style", "KEYWORD_ONLY", "gpt-j")]
    assert parameters(jax_ffi.apply_rotary_embedding) == [
        ("query", "POSITIONAL_OR_KEYWORD", empty), ("key", "POSITIONAL_OR_KEYWORD", empty),
        ("position_ids", "POSITIONAL_OR_KEYWORD", empty), ("inv_freq", "POSITIONAL_OR_KEYWORD", empty),
        ("rope_style", "KEYWORD_ONLY", "gpt-j")]
    assert parameters(jax_ffi.rms_norm) == [
        ("x", "POSITIONAL_OR_KEYWORD", empty), ("scale", "POSITIONAL_OR_KEYWORD", empty),
        ("eps", "POSITIONAL_OR_KEYWORD", empty), ("compute_dtype", "POSITIONAL_OR_KEYWORD", empty)]
    assert parameters(jax_ffi.shifted_targets_and_weights) == [
        ("input_ids", "POSITIONAL_OR_KEYWORD", empty), ("attention_mask", "POSITIONAL_OR_KEYWORD", empty),
        ("segment_ids", "POSITIONAL_OR_KEYWORD", None), ("assistant_mask", "POSITIONAL_OR_KEYWORD", None),
        ("loss_mask", "POSITIONAL_OR_KEYWORD", None), ("labels", "POSITIONAL_OR_KEYWORD", None),
        ("ignore_index", "KEYWORD_ONLY", -100)]
    assert parameters(jax_ffi.pallas_fused_sparse_cross_entropy) == [
        ("logits", "POSITIONAL_OR_KEYWORD", empty), ("targets", "POSITIONAL_OR_KEYWORD", empty),
        ("weights", "POSITIONAL_OR_KEYWORD", empty), ("mesh", "KEYWORD_ONLY", empty)]
    assert jax_ffi.AttentionMetadata._fields[:5] == (
        "query_segment_ids", "kv_segment_ids", "q_block_segments", "kv_block_segments", "attention_end")
    assert jax_ffi.AttentionMetadata._fields[5:] == ("tile_bounds",)
    # a frozen head asks XLA for a placeholder, not for a [d, V] gradient
    source = inspect.getsource(jax_ffi)
    assert "head.shape if lm_head_trainable else (8,)" in source and "np.float32(scale)" in source


def test_workload_generators_and_flop_accounting(ct):
    from oracle import attention_ref

    W = ct.workloads
    config = W.ATTENTION_CONFIGS["packed_small"]
    inputs = W.make_attention_inputs(config)
    ids = inputs["segment_ids"].numpy()
    assert ids.shape == (2, 1024) and inputs["q"].shape == (2, 1024, 8, 64)
    np.testing.assert_array_equal(attention_ref.canonicalize_segment_ids(ids != 0, ids), ids)
    pairs = W.count_allowed_pairs(ids)
    assert pairs == attention_ref.count_allowed_pairs(ids)
    assert W.attention_flops(config, pairs)["total"] == 14 * 64 * 8 * pairs
    rng = np.random.default_rng(0)
    seg, end = W.maskgit_layout(rng, 1, 4096)
    assert W.count_allowed_pairs(seg, end) == attention_ref.count_allowed_pairs(seg, end)
    blocks = np.flatnonzero(end[0] != np.arange(4096))
    assert len(blocks) % 1055 == 0 and len(blocks) > 0  # the last token of a block keeps end == itself
    cfg = W.CUTCE_CONFIGS["llama3_8b_head"]
    assert W.cutce_flops(cfg, 16384)["total"] == 6 * 16384 * 4096 * 128256
    assert W.attention_delta_bytes(W.ATTENTION_CONFIGS["llama3_8b"]) == 2 * 4 * 4096 * 32 * 128 * 2 + 4 * 4 * 4096 * 32
