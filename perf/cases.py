"""Performance cases: what a training or evaluation program has this package do, over the sizes it does it at.

Six kinds, each through the package's public entry points:

``batch``      once per batch: canonical segment ids, position ids, rotary tables, shifted targets and
               loss weights, attention metadata
``attention``  one layer's attention, forward and backward, from metadata that the batch keeps
``evaluate``   the same forward alone, without gradients
``layer``      the neighbours of attention in a decoder layer: RMS norm and rotary embedding, both directions
``cut_ce``     the loss from hidden states and the LM head, forward and backward
``sparse_ce``  the loss from logits that the caller has, forward and backward

The named sizes are those of the package's workloads, benchmark and tests; the others are generic.
A case fixes the lengths of the packed documents, the seed their order and all values: every
seed of a case is another batch with the same amount of work.
"""

import random

import torch

import causal_trainer_dev_amd as ct

_IMAGE = 32 * 33          # an image block: 32 rows of 32 codes and a line break


def listed():
    return [
        # The preparation of one batch of packed chat documents, at the size of the next case but one.
        dict(name="batch_4x4096", kind="batch", batch=4, seq=4096, shortest=64, longest=4096, images=False,
             q_heads=32, kv_heads=8, head_dim=128, rotary_dim=64),
        # A small model: short rows, heads of 64, every call a few microseconds of GPU work.
        dict(name="attention_packed_small", kind="attention", batch=2, seq=1024, q_heads=8, kv_heads=8, head_dim=64,
             shortest=32, longest=512, images=False, shared_workspace=False),
        # A layer of an 8B model over a packed batch; its layers share the backward's scratch.
        dict(name="attention_llama3_8b", kind="attention", batch=4, seq=4096, q_heads=32, kv_heads=8, head_dim=128,
             shortest=64, longest=4096, images=False, shared_workspace=True),
        # Text with image blocks that are bidirectional inside (per-query visible ends), no grouped heads.
        dict(name="attention_maskgit", kind="attention", batch=2, seq=8192, q_heads=16, kv_heads=16, head_dim=128,
             shortest=0, longest=0, images=True, shared_workspace=False),
        # Long context: a layer of a 70B model over one row of 32768 positions.
        dict(name="attention_long_70b", kind="attention", batch=1, seq=32768, q_heads=64, kv_heads=8, head_dim=128,
             shortest=512, longest=32768, images=False, shared_workspace=True),
        # Evaluation of a held-out batch: forward only, a row length that is no power of two, groups of three heads.
        dict(name="evaluate_3x2944", kind="evaluate", batch=3, seq=2944, q_heads=24, kv_heads=8, head_dim=64,
             shortest=40, longest=2944, images=False),
        # The neighbours of attention for a handful of tokens: latency and launches.
        dict(name="layer_small", kind="layer", batch=2, seq=130, hidden=1024, q_heads=8, kv_heads=2, head_dim=64,
             rotary_dim=32, style="gpt-neox", fused_scale=False),
        # The same at the 8B layer's size: passes over memory.
        dict(name="layer_llama3_8b", kind="layer", batch=4, seq=4096, hidden=4096, q_heads=32, kv_heads=8, head_dim=128,
             rotary_dim=64, style="gpt-j", fused_scale=True),
        # The loss of a small fine-tuning batch: an odd vocabulary, rows that fill no tile, nothing kept
        # between the two directions and no compaction.
        dict(name="cut_ce_small", kind="cut_ce", batch=3, seq=333, hidden=1024, vocab=32003, ignored=0.1, compaction=False,
             logits_cache=False, trainable=True, chunk=0, layout="dv"),
        # The loss of the 8B model: three tokens of ten are ignored (prompts), head of 128256 columns.
        dict(name="cut_ce_llama3_8b", kind="cut_ce", batch=4, seq=4096, hidden=4096, vocab=128256, ignored=0.3,
             compaction=True, logits_cache=True, trainable=True, chunk=0, layout="dv"),
        # The loss from f32 logits of a small model, odd in both sizes.
        dict(name="sparse_ce_f32_small", kind="sparse_ce", batch=3, seq=333, vocab=32003, ignored=0.1, dtype="float32"),
        # The loss from bf16 logits of the 8B model.
        dict(name="sparse_ce_llama3_8b", kind="sparse_ce", batch=4, seq=4096, vocab=128256, ignored=0.3, dtype="bfloat16"),
    ]


# ---------------------------------------------------------------------------------------- drawn cases

def _log(rng, low, high):
    """A whole number from `low` to `high`, even over its logarithm."""

    return min(high, max(low, round(low * (high / low) ** rng.random())))


def _rows(rng, low, high):
    """Rows of a batch and their length: `low` to `high` positions in all."""

    total = _log(rng, low, high)
    batch = rng.choice([b for b in (1, 2, 3, 4, 6, 8) if b <= total])
    return batch, max(1, total // batch)


def _packing(rng, most, images):
    """Batch, row length (a multiple of 128, as the attention operator takes it) and document lengths."""

    total = _log(rng, max(256, 2048 if images else 0), most)
    batch = rng.choice([b for b in (1, 2, 3, 4, 6, 8) if total // b >= (2048 if images else 128)])
    seq = max(1, total // batch // 128) * 128
    shortest = min(_log(rng, 16, 512), seq)
    return dict(batch=batch, seq=seq, shortest=0 if images else shortest,
                longest=0 if images else _log(rng, shortest, seq), images=images)


def _heads(rng):
    kv = rng.choice((1, 2, 4, 8, 16))
    return dict(q_heads=min(64, kv * rng.choice((1, 2, 3, 4, 6, 8))) // kv * kv, kv_heads=kv,
                head_dim=rng.choice((64, 128)))


def draw(rng):
    """One more case: the kinds as often as the list has them, sizes over the whole range of the kind."""

    largest = {c["name"]: c for c in listed()}
    while True:
        kind = rng.choice([c["kind"] for c in largest.values()])
        if kind == "batch":
            case = dict(_packing(rng, 32768, rng.random() < 0.25), **_heads(rng))
            case.update(kind=kind, rotary_dim=rng.choice((case["head_dim"], case["head_dim"] // 2)))
            return case
        if kind in ("attention", "evaluate"):
            case = dict(_packing(rng, 32768, rng.random() < 0.25), **_heads(rng), kind=kind)
            if kind == "attention":
                case["shared_workspace"] = rng.random() < 0.5
            if work(case)["flops"] <= 0.9 * work(largest["attention_long_70b"])["flops"]:
                return case
        if kind == "layer":
            batch, seq = _rows(rng, 4, 16384)
            heads = _heads(rng)
            case = dict(heads, kind=kind, batch=batch, seq=seq, hidden=8 * _log(rng, 16, 1024), style=rng.choice(("gpt-j", "gpt-neox")),
                        rotary_dim=rng.choice((heads["head_dim"], heads["head_dim"] // 2)), fused_scale=rng.random() < 0.5)
            if rng.random() < 0.5:      # the hidden sizes that models have
                case["hidden"] = rng.choice((512, 768, 1024, 2048, 2560, 4096, 5120, 8192))
            return case
        if kind == "cut_ce":
            batch, seq = _rows(rng, 64, 16384)
            case = dict(kind=kind, batch=batch, seq=seq, hidden=128 * _log(rng, 2, 64), vocab=_log(rng, 500, 185600),
                        ignored=round(0.9 * rng.random(), 2), compaction=rng.random() < 0.7, logits_cache=rng.random() < 0.6,
                        trainable=rng.random() < 0.8, chunk=0, layout="vd" if rng.random() < 0.15 else "dv")
            if rng.random() < 0.2:
                case["chunk"] = _log(rng, 16, max(16, batch * seq // 2))
            cost = batch * seq * case["hidden"] * case["vocab"]
            if cost <= 0.45 * 16384 * 4096 * 128256:
                return case
        if kind == "sparse_ce":
            batch, seq = _rows(rng, 4, 16384)
            case = dict(kind=kind, batch=batch, seq=seq, vocab=_log(rng, 500, 185600), ignored=round(0.9 * rng.random(), 2),
                        dtype=rng.choice(("bfloat16", "float32")))
            if batch * seq * case["vocab"] * (4 if case["dtype"] == "float32" else 2) <= 4 << 30:
                return case


# ---------------------------------------------------------------------------------------- inputs

def _documents(case):
    """The documents of each batch row as lists of (length, is an image) pieces; what does not fit is padding."""

    rng = random.Random("%(batch)d %(seq)d %(shortest)d %(longest)d %(images)d" % case)
    rows = []
    for _ in range(case["batch"]):
        row, used = [], 0
        while used < case["seq"]:
            if case["images"]:
                pieces = []
                for _ in range(rng.randint(1, 3)):
                    pieces += [(rng.randint(16, 256), False), (_IMAGE, True)]
                pieces.append((rng.randint(16, 128), False))
            else:
                pieces = [(_log(rng, case["shortest"], case["longest"]), False)]
            length = sum(size for size, _ in pieces)
            if used + length > case["seq"]:
                if row:
                    break
                pieces, length = [(case["seq"] - used, False)], case["seq"] - used
            row.append(pieces)
            used += length
        rows.append(row)
    return rows


def _pairs(case):
    """Visible (query, key) pairs: causal inside a document, an image's positions to the end of the image."""

    total = 0
    for row in _documents(case):
        for pieces in row:
            position = 0
            for size, image in pieces:
                total += size * (position + size) if image else size * position + size * (size + 1) // 2
                position += size
    return total


def _segments(case, seed):
    """Segment ids and inclusive visible ends `[batch, seq]` on the GPU, the documents in the seed's order."""

    rng, ids, ends = random.Random(seed), [], []
    for row in _documents(case):
        row = list(row)
        rng.shuffle(row)
        row_ids, row_ends = [], []
        for label, pieces in enumerate(row, 1):
            for size, image in pieces:
                at = len(row_ids)
                row_ids += [label] * size
                row_ends += [at + size - 1] * size if image else range(at, at + size)
        used = len(row_ids)
        ids.append(row_ids + [0] * (case["seq"] - used))
        ends.append(list(row_ends) + list(range(used, case["seq"])))
    as_device = lambda rows: torch.tensor(rows, dtype=torch.int32).cuda()  # noqa: E731
    return as_device(ids), as_device(ends) if case["images"] else None


def _profile(case):
    shape = lambda heads: (case["batch"], case["seq"], heads, case["head_dim"])  # noqa: E731
    return ct.resolve_attention_profile(shape(case["q_heads"]), shape(case["kv_heads"]), None, has_attention_end=case["images"])


def _loss_rows(case, generator, vocab):
    """Targets and weights of the loss: ignored positions have weight 0 and target -100."""

    shape = (case["batch"], case["seq"])
    targets = torch.randint(vocab, shape, generator=generator, device="cuda", dtype=torch.int32)
    order = torch.rand(shape, generator=generator, device="cuda").flatten().argsort()
    weights = torch.ones(shape, device="cuda")
    weights.view(-1)[order[:round(case["ignored"] * targets.numel())]] = 0
    return torch.where(weights > 0, targets, -100).to(torch.int32), weights


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0, dtype=torch.bfloat16):
        return torch.randn(shape, generator=generator, device="cuda", dtype=dtype).mul_(scale)

    kind, batch, seq = case["kind"], case["batch"], case["seq"]
    state = dict(case)
    if kind in ("batch", "attention", "evaluate"):
        segments, ends = _segments(case, seed)
        state["profile"] = _profile(case)
    if kind in ("attention", "evaluate", "layer"):
        state.update(q=normal(batch, seq, case["q_heads"], case["head_dim"]), k=normal(batch, seq, case["kv_heads"], case["head_dim"]))
    if kind == "batch":
        state.update(segments=segments, ends=ends, mask=(segments > 0).to(torch.int32),
                     tokens=torch.randint(128256, (batch, seq), generator=generator, device="cuda", dtype=torch.int32),
                     assistant=(torch.rand((batch, seq), generator=generator, device="cuda") < 0.7).to(torch.int32),
                     inv_freq=1e4 ** (-torch.arange(0, case["rotary_dim"], 2, dtype=torch.float32, device="cuda") / case["rotary_dim"]))
    elif kind in ("attention", "evaluate"):
        state.update(v=normal(batch, seq, case["kv_heads"], case["head_dim"]),
                     metadata=ct.prepare_attention_metadata(segments, mesh=None, profile=state["profile"], attention_end=ends))
        if kind == "attention":
            for name in "qkv":
                state[name].requires_grad_(True)
            state.update(dout=normal(batch, seq, case["q_heads"], case["head_dim"]),
                         workspace=ct.BackwardWorkspace() if case["shared_workspace"] else None)
    elif kind == "layer":
        positions = torch.arange(seq, dtype=torch.int32, device="cuda").repeat(batch, 1)
        inv_freq = 1e4 ** (-torch.arange(0, case["rotary_dim"], 2, dtype=torch.float32, device="cuda") / case["rotary_dim"])
        state["cosine"], state["sine"] = ct.rotary_cos_sin(positions, inv_freq)
        state.update(x=normal(batch, seq, case["hidden"]), scale=(1 + normal(case["hidden"], scale=0.1)),
                     dy=normal(batch, seq, case["hidden"]), dq=normal(batch, seq, case["q_heads"], case["head_dim"]),
                     dk=normal(batch, seq, case["kv_heads"], case["head_dim"]),
                     q_scale=case["head_dim"] ** -0.5 if case["fused_scale"] else 1.0)
        for name in ("x", "scale", "q", "k"):
            state[name].requires_grad_(True)
    elif kind == "cut_ce":
        head = (case["hidden"], case["vocab"]) if case["layout"] == "dv" else (case["vocab"], case["hidden"])
        state.update(x=normal(batch, seq, case["hidden"]), head=normal(*head, scale=0.02))
        state["targets"], state["weights"] = _loss_rows(case, generator, case["vocab"])
        state["dy"] = 1 / state["weights"].sum().clamp(min=1)
        state["x"].requires_grad_(True)
        state["head"].requires_grad_(case["trainable"])
    else:
        state["logits"] = normal(batch, seq, case["vocab"], scale=2.0, dtype=getattr(torch, case["dtype"])).requires_grad_(True)
        state["targets"], state["weights"] = _loss_rows(case, generator, case["vocab"])
        state["dy"] = (1 / state["weights"].sum().clamp(min=1)).expand(batch, seq).contiguous()
    return state


# ---------------------------------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "batch":
        canonical = ct.canonicalize_segment_ids(state["mask"], state["segments"])
        positions = ct.make_position_ids(state["mask"], state["segments"])
        cosine, sine = ct.rotary_cos_sin(positions, state["inv_freq"])
        targets, weights = ct.shifted_targets_and_weights(state["tokens"], state["mask"], state["segments"], state["assistant"])
        metadata = ct.prepare_attention_metadata(canonical, mesh=None, profile=state["profile"], attention_end=state["ends"])
        return dict(canonical=canonical, positions=positions, cosine=cosine, sine=sine, targets=targets, weights=weights,
                    queries=metadata.q_block_segments, keys=metadata.kv_block_segments, tiles=ct.tile_bounds_table(metadata))
    if kind == "evaluate":
        with torch.no_grad():
            return ct.efficient_attention(state["q"], state["k"], state["v"], state["metadata"], profile=state["profile"])
    if kind == "attention":
        inputs = (state["q"], state["k"], state["v"])
        out = ct.efficient_attention(*inputs, state["metadata"], profile=state["profile"], backward_workspace=state["workspace"])
        return out.detach(), *torch.autograd.grad(out, inputs, state["dout"])
    if kind == "layer":
        y = ct.rms_norm(state["x"], state["scale"], 1e-6)
        q, k = ct.apply_rotary_cos_sin(state["q"], state["k"], state["cosine"], state["sine"], rope_style=state["style"],
                                       q_scale=state["q_scale"])
        gradients = torch.autograd.grad((y, q, k), (state["x"], state["scale"], state["q"], state["k"]),
                                        (state["dy"], state["dq"], state["dk"]))
        return y.detach(), q.detach(), k.detach(), *gradients
    if kind == "cut_ce":
        nll, weight = ct.pallas_cut_linear_cross_entropy(
            state["x"], state["head"], state["targets"], state["weights"], sparse_compaction=state["compaction"],
            lm_head_trainable=state["trainable"], local_chunk_size=state["chunk"], logits_cache=state["logits_cache"],
            head_layout=state["layout"])
        inputs = (state["x"], state["head"]) if state["trainable"] else (state["x"],)
        return nll.detach(), weight, *torch.autograd.grad(nll, inputs, state["dy"])
    loss = ct.pallas_fused_sparse_cross_entropy(state["logits"], state["targets"], state["weights"])
    return loss.detach(), *torch.autograd.grad(loss, state["logits"], state["dy"])


# ---------------------------------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind, tokens = case["kind"], case["batch"] * case["seq"]
    if kind == "batch":
        # in: mask, segments, tokens, assistant mask (and ends); out: canonical ids, positions, targets, weights, two
        # tables in bf16, and the 12 integers of each block of 32 positions
        return {"bytes": tokens * (4 * (8 + case["images"]) + 2 * case["rotary_dim"] + 12 * 4 / 32), "flops": 0}
    if kind in ("attention", "evaluate"):
        unit = case["head_dim"] * case["q_heads"] * _pairs(case)
        rows, kv_rows = tokens * case["q_heads"], tokens * case["kv_heads"]
        forward = 2 * case["head_dim"] * (2 * rows + 2 * kv_rows)                      # q, out; k, v
        if kind == "evaluate":
            return {"bytes": forward, "flops": 4 * unit}
        # the backward reads q, out, dout, k, v and the row statistics and writes dq, dk, dv
        return {"bytes": forward + 2 * case["head_dim"] * (4 * rows + 4 * kv_rows) + 8 * rows, "flops": 14 * unit}
    if kind == "layer":
        # norm: x, y; x, dy, dx. rotary: both sides of q and k and the tables, once each way
        rotated = 4 * tokens * (case["q_heads"] + case["kv_heads"]) * case["head_dim"] + 2 * tokens * case["rotary_dim"]
        return {"bytes": 2 * tokens * case["hidden"] * 5 + 2 * rotated, "flops": 0}
    counted = tokens - round(case["ignored"] * tokens)
    if kind == "cut_ce":
        gemms = 3 if case["trainable"] else 2
        once = 2 * (tokens * case["hidden"] + case["hidden"] * case["vocab"])          # x, head
        back = 2 * tokens * case["hidden"] + (2 * case["hidden"] * case["vocab"] if case["trainable"] else 0)
        return {"bytes": 2 * once + back, "flops": 2 * gemms * counted * case["hidden"] * case["vocab"]}
    size = 4 if case["dtype"] == "float32" else 2
    return {"bytes": size * case["vocab"] * (2 * counted + tokens) + 16 * tokens, "flops": 0}


def tolerance(case):
    if case["kind"] == "batch":
        return {"rel": 4e-3}          # the tables: one rounding to bf16; everything else is whole numbers, or weights of 0 and 1
    if case["kind"] == "sparse_ce" and case["dtype"] == "float32":
        return {"rel": 1e-5}
    return {"rel": 1e-2}              # bf16 results of f32 sums over bf16 products
