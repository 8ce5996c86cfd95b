"""GPU parity of the cut cross-entropy hot path (through the C ABI) against oracle/cutce_ref.py.

Tolerances are the stated ones: scalar loss relative error <= 1e-4, dHidden / dHead relative
L2 <= 2e-2; the ignored-token set is exact (lse and dHidden are bitwise zero on ignored rows).
"""

import numpy as np
import pytest
import torch

from oracle import cutce_ref as ref
from oracle.attention_ref import relative_l2

pytestmark = pytest.mark.gpu

LOSS_RTOL, GRAD_RTOL, LSE_ATOL = 1e-4, 2e-2, 1e-3


def _bf16(array):
    return torch.from_numpy(np.asarray(array, dtype=np.float32)).to(torch.bfloat16)


def _case(seed, rows, width, vocab, pattern="random", hidden_scale=1.0, head_scale=0.05):
    rng = np.random.default_rng(seed)
    hidden = _bf16(rng.normal(scale=hidden_scale, size=(rows, width)))
    head = _bf16(rng.normal(scale=head_scale, size=(width, vocab)))
    targets = rng.integers(vocab, size=rows).astype(np.int32)
    weights = rng.choice(np.asarray([0.25, 1.0, 2.0], np.float32), size=rows).astype(np.float32)
    position = np.arange(rows)
    if pattern == "random":
        weights[rng.random(rows) < 0.3] = 0
    elif pattern == "trailing":
        weights[position >= rows // 3] = 0
    elif pattern == "alternating":
        weights[position % 2 == 1] = 0
    elif pattern == "middle":
        weights[(position < rows // 3) | (position >= rows // 2)] = 0
    elif pattern == "inactive":
        weights[:] = 0
    targets[weights == 0] = -100     # raw ignore labels do reach the kernel on zero-weight rows
    return hidden, head, torch.from_numpy(targets), torch.from_numpy(weights)


def _gpu(ct, device, hidden, head, targets, weights, dy, *, compaction, trainable=True, workspace=None,
         cache=False):
    hd, wd, td, ws = hidden.to(device), head.to(device), targets.to(device), weights.to(device)
    logits_cache = None
    if cache:
        size = ct.cut_cross_entropy.logits_cache_bytes(hidden.shape[0], hidden.shape[1], head.shape[1])
        # poisoned: every logit the backward uses must have been written by the forward
        logits_cache = torch.full((size,), 0xFF, dtype=torch.uint8, device=device)
    nll, weight_sum, lse = ct.cutce_forward(hd, wd, td, ws, sparse_compaction=compaction,
                                            logits_cache=logits_cache)
    dhidden, dhead = ct.cutce_backward(hd, wd, td, ws, lse, torch.tensor(dy), sparse_compaction=compaction,
                                       lm_head_trainable=trainable, workspace_bytes=workspace,
                                       logits_cache=logits_cache)
    torch.cuda.synchronize()
    return float(nll), float(weight_sum), lse.cpu(), dhidden.cpu(), None if dhead is None else dhead.cpu()


def _check(results, hidden, head, targets, weights, dy):
    nll, weight_sum, lse, dhidden, dhead = results
    nll_ref, weight_ref, lse_ref = ref.cut_forward(hidden, head, targets, weights)
    assert nll == pytest.approx(float(nll_ref), rel=LOSS_RTOL, abs=1e-6)
    assert weight_sum == float(weight_ref)
    assert float((lse - lse_ref).abs().max()) <= LSE_ATOL
    ignored = weights == 0
    assert (lse[ignored] == 0).all() and (lse[~ignored] != 0).all()     # identical ignored-token set
    assert (dhidden[ignored] == 0).all()
    dh_ref, dw_ref = ref.cut_backward(hidden, head, targets, weights, lse_ref, dy)
    assert relative_l2(dhidden, dh_ref) <= GRAD_RTOL
    if dhead is not None:
        assert relative_l2(dhead, dw_ref) <= GRAD_RTOL
    # and against the pure path (materialised logits + autograd)
    _, dh_pure, dw_pure = ref.full_logits_loss_and_grads(hidden, head, targets, weights, dy)
    assert relative_l2(dhidden, dh_pure) <= GRAD_RTOL
    if dhead is not None:
        assert relative_l2(dhead, dw_pure) <= GRAD_RTOL


@pytest.mark.parametrize("rows,width,vocab", [(256, 128, 256), (300, 128, 258), (1000, 256, 1500),
                                              (513, 384, 1031), (64, 128, 40)])
@pytest.mark.parametrize("compaction", [True, False])
@pytest.mark.parametrize("cache", [False, True])
def test_forward_backward_match_oracle(ct, gpu, rows, width, vocab, compaction, cache):
    print("case", rows, width, vocab, compaction, cache, flush=True)
    case = _case(rows + vocab, rows, width, vocab)
    _check(_gpu(ct, gpu, *case, 0.37, compaction=compaction, cache=cache), *case, 0.37)


def test_cached_logits_give_the_recomputed_gradients(ct, gpu):
    # the cache holds the same f32 logits the recomputation produces, so G and both gradients
    # agree to the last bit; also through the slab walk of a small workspace
    case = _case(21, 900, 256, 1500)
    plain = _gpu(ct, gpu, *case, 0.5, compaction=True)
    cached = _gpu(ct, gpu, *case, 0.5, compaction=True, cache=True)
    assert plain[0] == cached[0] and torch.equal(plain[2], cached[2])
    assert torch.equal(plain[3], cached[3]) and torch.equal(plain[4], cached[4])
    import ctypes
    shape = ct._lib.CutceShape(900, 256, 1500)
    least = ct._lib.load().ct_cutce_bwd_workspace_min_bytes(ctypes.byref(shape))
    slabs = _gpu(ct, gpu, *case, 0.5, compaction=True, cache=True, workspace=least)
    _check(slabs, *case, 0.5)
    assert torch.equal(slabs[4], cached[4])


@pytest.mark.parametrize("pattern", ["trailing", "alternating", "middle", "inactive"])
def test_weight_patterns(ct, gpu, pattern):
    # reference: tests/kernels/test_cross_entropy_tpu.py:166-239
    case = _case(7, 700, 128, 300, pattern)
    with_c = _gpu(ct, gpu, *case, 1.0, compaction=True)
    without = _gpu(ct, gpu, *case, 1.0, compaction=False)
    _check(with_c, *case, 1.0)
    _check(without, *case, 1.0)
    assert with_c[0] == pytest.approx(without[0], rel=1e-6, abs=1e-6) and with_c[1] == without[1]
    if pattern == "inactive":
        # reference: tests/kernels/test_tiled_cut.py:138-155
        assert with_c[0] == 0 and with_c[1] == 0
        assert not with_c[3].any() and not with_c[4].any()


@pytest.mark.parametrize("rows,cols", [(1, 128), (63, 128), (64, 64), (65, 200), (137, 77), (700, 384)])
def test_transpose16(ct, gpu, rows, cols):
    """The transposed copy of a [vocab, hidden] head: whole tiles, ragged ones, rows at odd addresses."""

    source = torch.randint(-2 ** 15, 2 ** 15, (rows, cols), dtype=torch.int16, device=gpu)
    copy = torch.empty((cols, rows), dtype=torch.int16, device=gpu)
    ct._lib.check(ct._lib.load().ct_transpose16(torch.cuda.current_stream().cuda_stream, source.data_ptr(), rows, cols,
                                                copy.data_ptr()))
    assert torch.equal(copy, source.t())


def test_small_hidden_large_logits_match_with_and_without_cache(ct, gpu):
    """Where the operator does without the logits cache (hidden sizes up to 768) the results
    are those of the recomputing form: the same f32 logits of the same products."""

    hidden, head, targets, weights = _case(9, 1100, 128, 65537)
    arguments = (targets.reshape(2, 550).to(gpu), weights.reshape(2, 550).to(gpu))
    outcomes = []
    for cache in (True, False):
        x, w = hidden.reshape(2, 550, 128).to(gpu).requires_grad_(True), head.to(gpu).requires_grad_(True)
        nll, _ = ct.pallas_cut_linear_cross_entropy(x, w, *arguments, logits_cache=cache)
        outcomes.append((nll.detach(), *torch.autograd.grad(nll, (x, w))))
    assert all(torch.equal(a, b) for a, b in zip(*outcomes))


@pytest.mark.parametrize("ignored", [0.0, 0.4, 1.0])
def test_operator_leaves_ignored_rows_out(ct, gpu, ignored):
    """The operator's results do not depend on sparse_compaction, and agree with the full-logits oracle."""

    hidden, head, targets, weights = _case(13, 300, 128, 501)
    targets = targets.clamp(min=0)     # (rows that _case ignores count here)
    weights = torch.where(torch.rand(300, generator=torch.Generator().manual_seed(3)) < ignored, 0.0, 1.0)
    arguments = (targets.reshape(1, 300).to(gpu), weights.reshape(1, 300).to(gpu))
    outcomes = []
    for compaction in (False, True):
        x, w = hidden.reshape(1, 300, 128).to(gpu).requires_grad_(True), head.to(gpu).requires_grad_(True)
        nll, total = ct.pallas_cut_linear_cross_entropy(x, w, *arguments, sparse_compaction=compaction)
        outcomes.append((nll.detach(), total, *torch.autograd.grad(nll, (x, w))))
    assert all(torch.equal(a, b) for a, b in zip(*outcomes))
    assert float(outcomes[0][1]) == float(weights.sum())
    if ignored < 1:
        _, dh_pure, dw_pure = ref.full_logits_loss_and_grads(hidden, head, targets, weights, 1.0)
        assert relative_l2(outcomes[0][2].cpu().reshape(300, 128), dh_pure) <= GRAD_RTOL
        assert relative_l2(outcomes[0][3].cpu(), dw_pure) <= GRAD_RTOL
    else:
        assert not outcomes[0][2].any() and not outcomes[0][3].any() and float(outcomes[0][0]) == 0


@pytest.mark.parametrize("cache", [False, True], ids=["recompute", "cache"])
def test_hidden_states_beyond_4_gib(ct, gpu, cache):
    """Active rows on both sides of the 4 GiB that a 32-bit offset reaches (row 262144 at this width)."""

    rows, width, vocab = 262144 + 300, 8192, 40
    line = (1 << 32) // (2 * width)
    active = torch.cat([torch.arange(5), torch.arange(1000, line, 1000), torch.arange(line - 40, line + 150, 3),
                        torch.tensor([rows - 1])])
    hidden, head, targets, _ = _case(31, active.numel(), width, vocab, hidden_scale=0.5)
    targets, weights = targets.clamp(min=0), torch.linspace(0.5, 1.5, active.numel())
    x = torch.zeros((4, rows // 4, width), dtype=torch.bfloat16, device=gpu)
    at = active.to(gpu)
    x.view(rows, width)[at] = hidden.to(gpu)
    all_targets = torch.full((rows,), -100, dtype=torch.int32, device=gpu)
    all_weights = torch.zeros(rows, device=gpu)
    all_targets[at], all_weights[at] = targets.to(gpu), weights.to(gpu)
    x.requires_grad_(True)
    w = head.to(gpu).requires_grad_(True)
    nll, total = ct.pallas_cut_linear_cross_entropy(x, w, all_targets.view(4, -1), all_weights.view(4, -1),
                                                    sparse_compaction=True, logits_cache=cache)
    dx, dw = torch.autograd.grad(nll, (x, w))
    nll_ref, weight_ref, _ = ref.cut_forward(hidden, head, targets, weights)
    assert float(nll.detach()) == pytest.approx(float(nll_ref), rel=LOSS_RTOL)
    assert float(total) == pytest.approx(float(weight_ref), rel=1e-6)
    _, dh_pure, dw_pure = ref.full_logits_loss_and_grads(hidden, head, targets, weights, 1.0)
    dx = dx.view(rows, width)
    assert torch.equal(dx.any(dim=1).nonzero().flatten(), at)
    assert relative_l2(dx[at].cpu(), dh_pure) <= GRAD_RTOL
    assert relative_l2(dw.cpu(), dw_pure) <= GRAD_RTOL


def test_forward_mode_is_refused(ct, gpu):
    """The operators have no forward-mode derivative: a dual input raises instead of losing its tangent."""

    from torch.autograd import forward_ad
    hidden, head, targets, weights = _case(7, 64, 128, 300)
    x = hidden.reshape(1, 64, 128).to(gpu)
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises(RuntimeError):
            ct.pallas_cut_linear_cross_entropy(dual, head.to(gpu), targets.reshape(1, 64).to(gpu), weights.reshape(1, 64).to(gpu))
        with pytest.raises(RuntimeError):
            ct.rms_norm(dual, torch.ones(128, dtype=torch.bfloat16, device=gpu), 1e-6)


def test_head_layout_vocab_major(ct, gpu):
    """The operator with the head given as [V, d] (a checkpoint's layout): the same loss and hidden
    gradient as with [d, V], bit for bit (the kernels see the same transposed copy), and the head's
    gradient in the layout the head came in."""

    hidden, head, targets, weights = _case(5, 600, 128, 700)
    hidden3 = hidden.reshape(2, 300, 128).to(gpu).requires_grad_(True)
    targets2, weights2 = targets.reshape(2, 300).to(gpu), weights.reshape(2, 300).to(gpu)
    outcomes = {}
    for layout in ("dv", "vd"):
        kernel = (head if layout == "dv" else head.t().contiguous()).to(gpu).requires_grad_(True)
        nll, weight_sum = ct.pallas_cut_linear_cross_entropy(hidden3, kernel, targets2, weights2, head_layout=layout)
        (dh, dw) = torch.autograd.grad(nll, (hidden3, kernel))
        outcomes[layout] = (float(nll.detach()), float(weight_sum.detach()), dh.cpu(), dw.cpu())
    assert outcomes["dv"][:2] == outcomes["vd"][:2]
    assert torch.equal(outcomes["dv"][2], outcomes["vd"][2])
    assert outcomes["vd"][3].shape == (700, 128) and torch.equal(outcomes["dv"][3], outcomes["vd"][3].t())
    _, dh_pure, dw_pure = ref.full_logits_loss_and_grads(hidden, head, targets, weights, 1.0)
    assert relative_l2(outcomes["vd"][2].reshape(600, 128), dh_pure) <= GRAD_RTOL
    assert relative_l2(outcomes["vd"][3].t(), dw_pure) <= GRAD_RTOL
    with pytest.raises(ValueError, match="head_layout"):
        ct.pallas_cut_linear_cross_entropy(hidden3, head.to(gpu), targets2, weights2, head_layout="rows")
    with pytest.raises(ValueError, match="hidden, vocab"):
        ct.pallas_cut_linear_cross_entropy(hidden3, head.to(gpu), targets2, weights2, head_layout="vd")


def test_small_workspace_walks_vocabulary_slabs(ct, gpu):
    case = _case(9, 900, 256, 1500)
    lib = ct._lib.load()
    shape = ct._lib.CutceShape(900, 256, 1500)
    import ctypes
    least = lib.ct_cutce_bwd_workspace_min_bytes(ctypes.byref(shape))
    full = lib.ct_cutce_bwd_workspace_bytes(ctypes.byref(shape))
    assert least < full
    one_slab = _gpu(ct, gpu, *case, 0.5, compaction=True)
    for workspace in (least, least + 2 * 1024 * 256 * 2):     # 1 and 3 tile columns per slab
        slabs = _gpu(ct, gpu, *case, 0.5, compaction=True, workspace=workspace)
        _check(slabs, *case, 0.5)
        assert torch.equal(slabs[4], one_slab[4])             # dHead does not depend on the slab walk
    with pytest.raises(ct._lib.CtError, match="workspace"):
        _gpu(ct, gpu, *case, 0.5, compaction=True, workspace=least - 256)


@pytest.mark.parametrize("rows,width,vocab,chunk", [(300, 256, 20001, 30), (84, 384, 9000, 22), (260, 128, 4097, 200),
                                                    (513, 128, 3000, 17)])
def test_slabs_leave_room_for_the_parts_of_dhidden(ct, gpu, rows, width, vocab, chunk):
    """A bounded workspace in slabs that are chosen by their time: few row blocks of long contractions, one slab without
    room for all parts, more row blocks."""

    case = _case(rows, rows, width, vocab)
    workspace = ct.cut_cross_entropy.backward_workspace_bytes(rows, width, vocab, chunk)
    one_slab = _gpu(ct, gpu, *case, 0.5, compaction=True)
    slabs = _gpu(ct, gpu, *case, 0.5, compaction=True, workspace=workspace)
    _check(slabs, *case, 0.5)
    assert torch.equal(slabs[4], one_slab[4])


@pytest.mark.parametrize("rows,width,vocab,chunk,trainable,slabs", [
    # 64 parts of dHidden fit behind one slab of the whole vocabulary, and no more are ever made
    (13, 256, 102429, 10, False, 1), (15, 128, 145924, 13, True, 1),
    # dHead's chains along the rows are walked once per slab; large partial sums
    (5542, 256, 23076, 698, True, 7), (5246, 1280, 12486, 2202, False, 2)])
def test_number_of_slabs_of_a_bounded_workspace(ct, gpu, rows, width, vocab, chunk, trainable, slabs):
    """The vocabulary is walked in no more slabs than is faster (the launches of a backward tell); a wider call's gradients."""

    hidden, head, targets, weights = (t.to(gpu) for t in _case(rows, rows, width, vocab))
    _, _, lse = ct.cutce_forward(hidden, head, targets, weights)
    workspace = ct.cut_cross_entropy.backward_workspace_bytes(rows, width, vocab, chunk)
    arguments = (hidden, head, targets, weights, lse, torch.ones(1))
    with ct.profiling.KernelTimer() as timer:
        bounded = ct.cutce_backward(*arguments, lm_head_trainable=trainable, workspace_bytes=workspace)
    assert len(timer.durations_ms()["cutce_dlogits_kernel"]) == slabs
    whole = ct.cutce_backward(*arguments, lm_head_trainable=trainable)
    assert relative_l2(bounded[0], whole[0]) <= 2.0 ** -8     # (f32 sums in another order, rounded to bf16 once)
    assert not trainable or torch.equal(bounded[1], whole[1])


def test_reference_seeded_fixture_and_frozen_head(ct, gpu):
    # inputs of the reference's tests/kernels/test_tiled_cut.py:66-128 (cotangent 0.37)
    golden = np.load("tests/golden/cutce_rng460.npz")
    hidden = torch.from_numpy(golden["hidden"]).view(torch.bfloat16)        # [2, 386, 128]
    head = torch.from_numpy(golden["head"]).view(torch.bfloat16)
    targets, weights = torch.from_numpy(golden["targets"]), torch.from_numpy(golden["weights"])
    hd = hidden.to(gpu).requires_grad_(True)
    wd = head.to(gpu).requires_grad_(True)
    for compaction in (False, True):
        hd.grad = wd.grad = None
        nll, weight_sum = ct.pallas_cut_linear_cross_entropy(hd, wd, targets.to(gpu), weights.to(gpu), mesh=None,
                                                             sparse_compaction=compaction)
        (nll * 0.37 + weight_sum * 0.0).backward()
        assert float(nll) == pytest.approx(float(golden["nll_sum"]), rel=2e-5, abs=2e-3)
        assert float(weight_sum) == float(golden["weight_sum"])
        expected_dh = torch.from_numpy(golden["dhidden"]).view(torch.bfloat16).reshape(hidden.shape)
        expected_dw = torch.from_numpy(golden["dhead"]).view(torch.bfloat16)
        assert relative_l2(hd.grad.cpu(), expected_dh) < GRAD_RTOL
        assert relative_l2(wd.grad.cpu(), expected_dw) < GRAD_RTOL
        assert (hd.grad.cpu()[weights == 0] == 0).all()
    # frozen head: no head gradient is produced at all (reference :645-667)
    hd.grad = wd.grad = None
    nll, _ = ct.pallas_cut_linear_cross_entropy(hd, wd, targets.to(gpu), weights.to(gpu), mesh=None,
                                                lm_head_trainable=False)
    nll.backward()
    assert wd.grad is None and hd.grad is not None
    with pytest.raises(ValueError, match="fsdp=ep=1"):
        ct.pallas_cut_linear_cross_entropy(hd, wd, targets.to(gpu), weights.to(gpu), mesh={"fsdp": 2})


@pytest.mark.parametrize("compaction,trainable", [(False, True), (True, True), (False, False)])
def test_chunked_option_against_the_chunk_loop_oracle(ct, gpu, compaction, trainable):
    # the one-device case of the reference's tests/kernels/test_tiled_cut.py:89-128:
    # chunks of 128 over 2 x 386 rows (ragged last chunk), cotangent 0.37
    from oracle import cutce_ref

    golden = np.load("tests/golden/cutce_rng460.npz")
    hidden = torch.from_numpy(golden["hidden"]).view(torch.bfloat16)
    head = torch.from_numpy(golden["head"]).view(torch.bfloat16)
    targets, weights = torch.from_numpy(golden["targets"]), torch.from_numpy(golden["weights"])
    flat = hidden.reshape(-1, 128)
    want_nll, want_weight, lse = cutce_ref.chunked_cut_forward(flat, head, targets.reshape(-1), weights.reshape(-1),
                                                               128, sparse_compaction=compaction)
    want_dh, want_dw = cutce_ref.chunked_cut_backward(flat, head, targets.reshape(-1), weights.reshape(-1), lse,
                                                      0.37, 128, head_trainable=trainable)
    hd = hidden.to(gpu).requires_grad_(True)
    wd = head.to(gpu).requires_grad_(True)
    nll, weight_sum = ct.pallas_cut_linear_cross_entropy(hd, wd, targets.to(gpu), weights.to(gpu), mesh=None,
                                                         sparse_compaction=compaction, lm_head_trainable=trainable,
                                                         local_chunk_size=128)
    (nll * 0.37 + weight_sum * 0.0).backward()
    assert float(nll) == pytest.approx(float(want_nll), rel=LOSS_RTOL)
    assert float(weight_sum) == float(want_weight)
    assert relative_l2(hd.grad.cpu().reshape(-1, 128), want_dh) < GRAD_RTOL
    assert (hd.grad.cpu()[weights == 0] == 0).all()
    if trainable:
        assert relative_l2(wd.grad.cpu(), want_dw) < GRAD_RTOL
    else:
        assert wd.grad is None


def test_chunk_size_shrinks_the_workspace_and_keeps_the_results(ct, gpu):
    """local_chunk_size bounds the backward's workspace (the dlogits slab covers as much as one
    chunk of rows would need) and changes nothing but the order of f32 additions."""

    from causal_trainer_dev_amd.cut_cross_entropy import backward_workspace_bytes

    rows, width, vocab = 1000, 256, 6000          # 24 vocabulary tiles
    hidden, head, targets, weights = _case(17, rows, width, vocab)
    full = backward_workspace_bytes(rows, width, vocab, 0)
    bounded = backward_workspace_bytes(rows, width, vocab, 250)
    assert bounded < 0.6 * full
    results = {}
    for chunk in (0, 250):
        hd = hidden.to(gpu).reshape(1, rows, width).requires_grad_(True)
        wd = head.to(gpu).requires_grad_(True)
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        nll, weight_sum = ct.pallas_cut_linear_cross_entropy(
            hd, wd, targets.to(gpu).reshape(1, rows), weights.to(gpu).reshape(1, rows), mesh=None,
            sparse_compaction=True, local_chunk_size=chunk, logits_cache=False)
        (nll * 0.5).backward()
        torch.cuda.synchronize()
        results[chunk] = (float(nll), float(weight_sum), hd.grad.cpu(), wd.grad.cpu(),
                          torch.cuda.max_memory_allocated() - before)
    whole, chunked = results[0], results[250]
    assert whole[0] == chunked[0] and whole[1] == chunked[1]
    assert relative_l2(chunked[2], whole[2]) < 1e-3 and relative_l2(chunked[3], whole[3]) < 1e-3
    assert whole[4] - chunked[4] >= (full - bounded) // 2      # the peak really is lower
    _, dh_ref, dw_ref = ref.full_logits_loss_and_grads(hidden, head, targets, weights, 0.5)
    assert relative_l2(chunked[2].reshape(rows, width), dh_ref) <= GRAD_RTOL
    assert relative_l2(chunked[3], dw_ref) <= GRAD_RTOL


def test_chunked_option_all_masked_rows_and_frozen_head(ct, gpu):
    # tests/kernels/test_tiled_cut.py:138-155
    golden = np.load("tests/golden/cutce_rng460.npz")
    hidden = torch.from_numpy(golden["hidden"]).view(torch.bfloat16)[:1, :199].contiguous()
    head = torch.from_numpy(golden["head"]).view(torch.bfloat16)
    hd = hidden.to(gpu).requires_grad_(True)
    wd = head.to(gpu).requires_grad_(True)
    targets = torch.full((1, 199), -100, dtype=torch.int32, device=gpu)
    nll, weight_sum = ct.pallas_cut_linear_cross_entropy(hd, wd, targets, torch.zeros(1, 199, device=gpu), mesh=None,
                                                         sparse_compaction=True, lm_head_trainable=False,
                                                         local_chunk_size=128)
    nll.backward()
    assert float(nll) == float(weight_sum) == 0.0
    assert wd.grad is None and not hd.grad.any()


def test_closed_form_uniform_logits(ct, gpu):
    # zero hidden => nll = sum(w) log V (reference: tests/training/test_losses.py:125-252)
    rows, vocab = 300, 1000
    hidden = torch.zeros((rows, 128), dtype=torch.bfloat16)
    head = _bf16(np.random.default_rng(0).normal(size=(128, vocab)))
    weights = torch.from_numpy(np.random.default_rng(1).choice([0.0, 0.25, 1.0], size=rows).astype(np.float32))
    targets = torch.arange(rows, dtype=torch.int32) % vocab
    nll, weight_sum, lse, dhidden, _ = _gpu(ct, gpu, hidden, head, targets, weights, 1.0, compaction=True)
    assert nll == pytest.approx(float(weights.sum()) * np.log(vocab), rel=1e-6)
    assert weight_sum == float(weights.sum())
    assert float((lse[weights != 0] - np.log(vocab)).abs().max()) < 1e-5


@pytest.mark.parametrize("cache", [False, True], ids=["recompute", "logits_cache"])
def test_benchmark_shape(ct, gpu, cache):
    """N=16384, d=4096, V=128256, 30% ignored: oracle on samples + size-independent properties,
    for the backward that recomputes the logits and for the one that reads the forward's f32
    logits cache (8.4 GB here, poisoned before the forward: offsets beyond 2^32 bytes)."""

    W = ct.workloads
    config = W.CUTCE_CONFIGS["llama3_8b_head"]
    inputs = W.make_cutce_inputs(config)
    hidden, head, targets, weights = (inputs[n] for n in ("hidden", "head", "targets", "weights"))
    active = int((weights != 0).sum())
    dy = 1.0 / active
    print("shape", config, "active", active, flush=True)
    nll, weight_sum, lse, dhidden, dhead = _gpu(ct, gpu, hidden, head, targets, weights, dy, compaction=True,
                                                cache=cache)
    assert weight_sum == float(active)
    ignored = weights == 0
    assert (lse[ignored] == 0).all() and (lse[~ignored] != 0).all()
    assert (dhidden[ignored] == 0).all()
    assert torch.isfinite(dhidden.float()).all() and torch.isfinite(dhead.float()).all()

    # rows: oracle on a sample of 512 rows (full vocabulary)
    rng = np.random.default_rng(0)
    sample = torch.from_numpy(np.sort(rng.choice(config.rows, size=512, replace=False)))
    head_f32 = head.float()
    logits = hidden[sample].float() @ head_f32
    lse_ref = torch.where(weights[sample] != 0, torch.logsumexp(logits, -1), 0.0)
    assert float((lse[sample] - lse_ref).abs().max()) <= LSE_ATOL
    dh_ref, _ = ref.cut_backward(hidden[sample], head, targets[sample], weights[sample], lse_ref, dy,
                                 head_trainable=False)
    assert relative_l2(dhidden[sample], dh_ref) <= GRAD_RTOL

    # scalar loss: f64 sum of per-row losses with the device lse (verified on the sample above)
    # and target logits recomputed on the host for every active row
    rows = torch.nonzero(~ignored).flatten()
    target_logit = (hidden[rows].float() * head_f32[:, targets[rows].long()].T).sum(-1).double()
    nll_ref = float(((lse[rows].double() - target_logit) * weights[rows].double()).sum())
    assert nll == pytest.approx(nll_ref, rel=LOSS_RTOL)

    # columns: dHead on 256 sampled vocabulary columns, G rebuilt on the host from the device lse
    cols = torch.from_numpy(np.sort(rng.choice(config.vocab, size=256, replace=False)))
    col_logits = hidden.float() @ head_f32[:, cols]
    prob = torch.where(~ignored[:, None], torch.exp(col_logits - lse[:, None]), 0.0)
    onehot = (targets[:, None].long() == cols[None, :]) & ~ignored[:, None]
    g = ((weights * dy)[:, None] * (prob - onehot.float())).to(torch.bfloat16).float()
    dw_ref = hidden.float().T @ g
    assert relative_l2(dhead[:, cols], dw_ref) <= GRAD_RTOL


@pytest.mark.parametrize("rows,width,vocab", [
    (1, 128, 7),          # smaller than any tile, one term in the last group
    (70, 1408, 1016),     # aligned rows, a ragged last tile, half a hidden tile; both gradients cut
    (999, 256, 4099),     # unaligned rows: the panel; dHidden cut
    (2817, 384, 264),     # many rows, two vocabulary tiles: dHead cut
    (513, 128, 33025),    # units of several vocabulary tiles, one column in the last
])
def test_ragged_sizes_and_cut_contractions(ct, gpu, rows, width, vocab):
    """Sizes at the edges of the panel, of the tiles and of the parts the gradient contractions are cut
    into; the forward gives the same bits whatever part of the panel its workspace holds."""

    import ctypes

    case = _case(rows + vocab, rows, width, vocab)
    for cache in (False, True):
        print("case", rows, width, vocab, cache, flush=True)
        _check(_gpu(ct, gpu, *case, 0.37, compaction=True, cache=cache), *case, 0.37)
    lib, shape = ct._lib.load(), ct._lib.CutceShape(rows, width, vocab)
    least = lib.ct_cutce_fwd_workspace_min_bytes(ctypes.byref(shape))
    full = lib.ct_cutce_fwd_workspace_bytes(ctypes.byref(shape))
    assert (full > least) == (vocab % 8 != 0)
    hidden, head, targets, weights = (t.to(gpu) for t in case)
    results = []
    for size in (full, (least + full) // 2, least):     # all of the panel, some of it, the guarded loop
        out = torch.full((rows + 2,), float("nan"), device=gpu)
        workspace = torch.empty(size, dtype=torch.uint8, device=gpu)
        args = ct._lib.CutceFwdArgs(
            hidden=hidden.data_ptr(), head=head.data_ptr(), targets=targets.data_ptr(), weights=weights.data_ptr(),
            nll_sum=out[0:].data_ptr(), weight_sum=out[1:].data_ptr(), lse=out[2:].data_ptr(),
            workspace=workspace.data_ptr(), workspace_bytes=size, shape=shape, sparse_compaction=1)
        ct._lib.check(lib.ct_cutce_fwd(ct._lib.current_stream(), args))
        results.append(out.cpu())
    assert all(torch.equal(r, results[0]) for r in results[1:]) and torch.isfinite(results[0]).all()


@pytest.mark.parametrize("rows,width,vocab", [
    (129, 128, 248),      # both products in 128 x 128 tiles, one column and one row past a tile
    (50, 4224, 520),      # rows longer than what is read ahead of the list
    (1024, 256, 6144),    # 8 x 48 small tiles, gradients in large ones
    (1025, 256, 5500),    # 9 x 43, unaligned rows
    (1024, 768, 4096),    # 8 x 32 small tiles, the most that have a compute unit each, 24 steps
    (1024, 768, 4104),    # 8 x 33
    (130, 896, 700),      # 2 x 6: a last half of eight steps; d = 640 below is too short for them
    (1024, 256, 7680),    # 8 x 60 small tiles: the last projection that takes them
    (1025, 256, 6912),    # 9 x 54: the first in large tiles, 5 x 27 of them: a round that fills part of the device
    (897, 640, 1288),     # gradients in small tiles, the last 8 columns from the tail
    (1025, 1152, 1288),   # small tiles for the projection, large ones for the gradients
    (1023, 2048, 300),    # row lists: four wavefronts a row, the last workgroup ragged
    (1030, 8192, 130),    # two, of rows longer than what is read ahead
    (4099, 128, 300),     # row lists: two rounds of 16 rows per workgroup, the last one ragged
    (70001, 128, 130),    # 18 rounds: five wavefronts list rows
])
def test_output_tile_sizes(ct, gpu, rows, width, vocab):
    """Sizes on both sides of the lines between the 128 x 128 and the 256 x 256 tiles and between the sizes of the
    backward's row lists, with and without the logits cache and compaction; dHead is the same for every workspace."""

    case = _case(rows + vocab, rows, width, vocab)
    for cache, compaction in ((False, True), (True, True), (False, False)):
        print("case", rows, width, vocab, cache, compaction, flush=True)
        _check(_gpu(ct, gpu, *case, 0.37, compaction=compaction, cache=cache), *case, 0.37)
    hidden, head, targets, weights = (t.to(gpu) for t in case)
    dy = torch.tensor(0.37, device=gpu)
    _, _, lse = ct.cutce_forward(hidden, head, targets, weights, sparse_compaction=True)
    whole = ct.cutce_backward(hidden, head, targets, weights, lse, dy, sparse_compaction=True)
    least = ct.cut_cross_entropy.backward_workspace_bytes(rows, width, vocab, 1)
    slabs = ct.cutce_backward(hidden, head, targets, weights, lse, dy, sparse_compaction=True, workspace_bytes=least)
    assert torch.equal(whole[1], slabs[1])
    assert relative_l2(slabs[0].cpu(), whole[0].cpu()) <= GRAD_RTOL


@pytest.mark.parametrize("rows,vocab", [(257, 128 * 64), (257, 128 * 65), (33, 128 * 64 + 1), (1, 16381)])
def test_merge_of_long_and_short_walks(ct, gpu, rows, vocab):
    """64 chunks of the vocabulary for a row, the most that 8 threads merge, and 65 and more, which 32 do."""

    _check(_gpu(ct, gpu, *_case(rows + vocab, rows, 128, vocab), 0.37, compaction=True), *_case(rows + vocab, rows, 128, vocab), 0.37)


@pytest.mark.parametrize("rows,width,vocab", [
    (4200, 128, 16380),   # four to five large tiles per workgroup of four steps each, unaligned rows
    (8500, 128, 20008),   # units of two tiles, the last of one
    (2100, 640, 16383),   # more steps than a tile's first iteration has
])
def test_tiles_one_after_the_other(ct, gpu, rows, width, vocab):
    """Workgroups that walk several tiles, each of whose first copies travel behind the epilogue of the tile before;
    the targets crowd the edges of tiles and of the wavefronts' parts of them, several of a wavefront's rows to one."""

    hidden, head, _, weights = _case(rows + vocab, rows, width, vocab)
    edges = torch.tensor([0, 3, 4, 127, 128, 255, 256, vocab - 257, vocab - 1], dtype=torch.int32)
    targets = edges[torch.randint(len(edges), (rows,), generator=torch.Generator().manual_seed(rows))]
    case = (hidden, head, targets, weights)
    for cache, compaction in ((False, True), (True, True), (False, False)):
        print("case", rows, width, vocab, cache, compaction, flush=True)
        _check(_gpu(ct, gpu, *case, 0.37, compaction=compaction, cache=cache), *case, 0.37)


@pytest.mark.parametrize("rows,width,vocab", [(300, 256, 1031), (70, 128, 7), (513, 1152, 4098)])
@pytest.mark.parametrize("layout,cache", [("dv", False), ("vd", False), ("vd", True)])
def test_one_aligned_copy_for_both_directions(ct, gpu, rows, width, vocab, layout, cache):
    """An unaligned head's copy that the forward leaves to the backward, or that is transposed into its place: the bits of
    the two calls that make a copy each, in a first backward and in a second one, which makes its own."""

    hidden, head, targets, weights = (t.to(gpu) for t in _case(rows + vocab, rows, width, vocab))
    dy = torch.tensor(0.37, device=gpu)
    nll, _, lse = ct.cutce_forward(hidden, head, targets, weights, sparse_compaction=True)
    dx, dw = ct.cutce_backward(hidden, head, targets, weights, lse, dy, sparse_compaction=True)
    x = hidden.view(1, rows, width).requires_grad_(True)
    w = (head if layout == "dv" else head.t().contiguous()).requires_grad_(True)
    got, _ = ct.pallas_cut_linear_cross_entropy(x, w, targets.view(1, -1), weights.view(1, -1), logits_cache=cache,
                                                head_layout=layout)
    assert torch.equal(got.detach(), nll)
    for last in (False, True):
        gx, gw = torch.autograd.grad(got, (x, w), dy, retain_graph=not last)
        assert torch.equal(gx.view(rows, width), dx)
        assert torch.equal(gw if layout == "dv" else gw.t(), dw)


@pytest.mark.parametrize("rows,width,vocab,both", [
    (64, 1536, 8209, True),     # small tiles in the projections; the last one is the tail's first half
    (100, 128, 96001, True),    # large projections, small tiles in the gradients
    (300, 1024, 12543, True),   # small tiles, the last one the tail's second half; a tail of 255 columns
    (500, 1024, 16250, True),   # large tiles; a tail of 122 columns, 4-byte aligned rows
    (1024, 1152, 10890, True),  # the most rows that both directions read in place, a tail of 138 columns
    (1025, 1152, 10891, False),  # one more: the forward only
    (1500, 256, 16001, False),  # a tail of 129 columns
    (513, 768, 32021, True),    # more parts of dHidden than tiles, the last of them the tail's
])
@pytest.mark.parametrize("cache,trainable", [(False, True), (True, True), (False, False)])
def test_head_read_in_place(ct, gpu, rows, width, vocab, both, cache, trainable):
    """An unaligned head of few rows, which the kernels read in place: the bits that its aligned copy gives, which a
    transposed head goes through, with and without the logits cache and with hidden rows that are unaligned themselves, and
    the f32 gradients."""

    shape = ct._lib.CutceShape(rows, width, vocab)
    assert ct._lib.load().ct_cutce_head_in_place(shape) == both
    case = _case(rows + vocab, rows, width, vocab)
    hidden, head, targets, weights = (t.to(gpu) for t in case)
    outcomes = []
    shifted = torch.empty(rows * width + 1, dtype=torch.bfloat16, device=gpu)[1:].copy_(hidden.flatten())
    for layout, source in (("dv", hidden), ("vd", hidden), ("dv", shifted)):
        x = source.detach().view(1, rows, width).requires_grad_(True)
        w = (head if layout == "dv" else head.t().contiguous()).requires_grad_(True)
        nll, _ = ct.pallas_cut_linear_cross_entropy(x, w, targets.view(1, -1), weights.view(1, -1), logits_cache=cache,
                                                    lm_head_trainable=trainable, head_layout=layout)
        grads = torch.autograd.grad(nll, (x, w) if trainable else (x,), torch.tensor(0.37, device=gpu))
        outcomes.append((nll.detach(), grads[0].view(rows, width), *(g if layout == "dv" else g.t() for g in grads[1:])))
    assert all(torch.equal(a, b) and torch.equal(a, c) for a, b, c in zip(*outcomes))
    x, w = hidden.float(), head.float()
    logits = x @ w
    lse = torch.logsumexp(logits, 1)
    g = torch.softmax(logits, 1)
    g[torch.arange(rows), targets.long().clamp(min=0)] -= 1
    g *= (0.37 * weights)[:, None]
    assert relative_l2(outcomes[0][1].cpu(), (g @ w.t()).cpu()) <= GRAD_RTOL
    if trainable:
        assert relative_l2(outcomes[0][2].cpu(), (x.t() @ g).cpu()) <= GRAD_RTOL
    picked = logits[torch.arange(rows), targets.long().clamp(min=0)]
    assert float(outcomes[0][0]) == pytest.approx(float((weights * (lse - picked)).double().sum()), rel=2e-5, abs=2e-3)


@pytest.mark.parametrize("rows,width,vocab,columns", [
    (64, 1536, 8209, 1),    # a slab for each tile column, the last one the tail's first half
    (300, 1024, 12543, 3),  # a last slab of one column
    (513, 768, 32021, 40),  # parts of dHidden that end inside of a slab
])
@pytest.mark.parametrize("trainable", [True, False])
def test_head_read_in_place_in_slabs(ct, gpu, rows, width, vocab, columns, trainable):
    """A bounded workspace: the vocabulary in slabs, the head in place all the same (no copy is made for a slab)."""

    import ctypes

    lib, shape = ct._lib.load(), ct._lib.CutceShape(rows, width, vocab)
    case = _case(rows + vocab, rows, width, vocab)
    least = lib.ct_cutce_bwd_workspace_min_bytes(ctypes.byref(shape))
    size = least + (columns - 1) * ((rows + 255) // 256 * 256) * 256 * 2
    assert size < lib.ct_cutce_bwd_workspace_used_bytes(ctypes.byref(shape))
    whole = _gpu(ct, gpu, *case, 0.37, compaction=True, trainable=trainable)
    with ct.profiling.KernelTimer() as timer:
        slabs = _gpu(ct, gpu, *case, 0.37, compaction=True, trainable=trainable, workspace=size)
    launches = timer.durations_ms()
    assert len(launches["cutce_dlogits_kernel"]) > 1 and len(launches["cutce_prepare_kernel"]) == 2  # (one a direction)
    assert relative_l2(slabs[3], whole[3]) <= 2.0 ** -8     # (f32 sums in another order, rounded to bf16 once)
    assert not trainable or torch.equal(slabs[4], whole[4])
    if trainable:
        _check(slabs, *case, 0.37)


@pytest.mark.parametrize("rows,cols,ld", [(7, 128, 256), (65, 64, 65), (1031, 200, 1280)])
def test_transpose16_into_padded_rows(ct, gpu, rows, cols, ld):
    source = torch.randint(-2 ** 15, 2 ** 15, (rows, cols), dtype=torch.int16, device=gpu)
    out = torch.full((cols, ld), 77, dtype=torch.int16, device=gpu)
    ct._lib.check(ct._lib.load().ct_transpose16_padded(torch.cuda.current_stream().cuda_stream, source.data_ptr(), rows, cols,
                                                       out.data_ptr(), ld))
    assert torch.equal(out[:, :rows], source.t()) and not out[:, rows:].any()
