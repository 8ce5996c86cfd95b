"""Generates ct_attn_asm.inc: hand-scheduled MFMA sequences of the attention kernels (D = 128).

The compiler's scheduler places every LDS fragment read directly in front of the MFMA that
consumes it once register pressure is high, so each MFMA pays the full LDS latency. These
sequences pin the order instead: fragment reads run AHEAD fragments in front of their MFMA,
into fixed scratch registers v[240:255] (declared as clobbers), and s_waitcnt lgkmcnt(n) is
exact because nothing else of the wavefront is counted by lgkmcnt while a sequence runs (each
starts with lgkmcnt(0)).

Run ``python gen_attn_asm.py > ct_attn_asm.inc`` after editing; the output is committed.
"""

SCRATCH0 = 240
# The compiler cannot see the MFMAs inside an asm statement, so it will not insert the wait
# states that a vector ALU read of a fresh MFMA result needs; the sequences end with them (the steps of dQ and dK/dV, whose sums
# stay in accumulation registers, leave them to whoever reads those).
TAIL = ["s_nop 15", "s_nop 7"]

def slot_regs(slot):
    lo = SCRATCH0 + 4 * slot
    return lo, lo + 3


def emit(lines, name):
    body = "\n".join('  "%s\\n\\t"' % ln for ln in lines)
    return "#define %s \\\n%s\n" % (name, body.replace("\n", " \\\n"))


def pv_sequence(ahead, slots):
    """O^T[db] += V^T frag(step, db) * P^T[step]: 16 MFMAs, each fragment = 2 ds_read_b64_tr_b16.

    operands: %0-%3 accumulators, %4-%7 lo pointers (column block db), %8-%11 hi pointers,
    %12-%15 probability fragments (k-step), %16 byte offset of the V tile.
    """
    n = 16
    lines = ["s_waitcnt lgkmcnt(0)"]

    def load(i):
        step, db = divmod(i, 4)
        lo, _ = slot_regs(i % slots)
        off = "%%16+%d" % (step * 4096)
        return ["ds_read_b64_tr_b16 v[%d:%d], %%%d offset:%s" % (lo, lo + 1, 4 + db, off),
                "ds_read_b64_tr_b16 v[%d:%d], %%%d offset:%s" % (lo + 2, lo + 3, 8 + db, off)]

    for i in range(min(ahead, n)):
        lines += load(i)
    for i in range(n):
        later = min(ahead - 1, n - 1 - i)
        lines.append("s_waitcnt lgkmcnt(%d)" % (2 * later))
        step, db = divmod(i, 4)
        lo, hi = slot_regs(i % slots)
        lines.append("v_mfma_f32_32x32x16_bf16 %%%d, v[%d:%d], %%%d, %%%d" % (db, lo, hi, 12 + step, db))
        if i + ahead < n:
            lines += load(i + ahead)
    return lines + TAIL


def qk_sequence(ahead, slots):
    """S^T[kb] = K frag(kb, ks) * Q^T[ks]: 16 MFMAs, each fragment = 1 ds_read_b128.

    operands: %0-%1 score accumulators (written), %2-%9 fragment pointers (k-step ks),
    %10-%17 query fragments (k-step), %18 byte offset of the K tile.
    """
    n = 16
    lines = ["s_waitcnt lgkmcnt(0)"]

    def load(i):
        ks, kb = divmod(i, 2)
        lo, hi = slot_regs(i % slots)
        return ["ds_read_b128 v[%d:%d], %%%d offset:%%18+%d" % (lo, hi, 2 + ks, kb * 8192)]

    for i in range(min(ahead, n)):
        lines += load(i)
    for i in range(n):
        later = min(ahead - 1, n - 1 - i)
        lines.append("s_waitcnt lgkmcnt(%d)" % later)
        ks, kb = divmod(i, 2)
        lo, hi = slot_regs(i % slots)
        src_c = "0" if ks == 0 else "%%%d" % kb
        lines.append("v_mfma_f32_32x32x16_bf16 %%%d, v[%d:%d], %%%d, %s" % (kb, lo, hi, 10 + ks, src_c))
        if i + ahead < n:
            lines += load(i + ahead)
    return lines + TAIL


# ---------------------------------------------------------------------------
# Forward, interleaved form. A wavefront that runs its softmax arithmetic and its MFMAs in
# separate stretches leaves the matrix pipe idle during the first and the vector ALU idle during
# the second; the other wavefront of the SIMD fills only part of that. Here the arithmetic of key
# tile t sits between the MFMAs of O += V(t-1)^T P(t-1)^T and S(t+1)^T = K(t+1) Q^T of the same
# wavefront: about five vector instructions fit behind an MFMA without delaying the next one.
#
# The scores live in two buffers of 32 registers that only these statements name, v[176:207] ("a")
# and v[208:239] ("b"); the compiler is kept out of v[176:255] (clobbers on every statement, and a
# static check of the compiled kernel). The scores of tile t are in buffer a when t counts even
# from the first tile of the query tile, else in b; S(t+1) is written to the other buffer while
# the exponentials of tile t are taken in place. The bf16 pairs of P(t) go into the first 16
# registers of the buffer they came from (pair p reads scores 2p, 2p+1 and writes register p, which
# an earlier pair has already read), where the PV product of the next step finds them; by the time
# S(t+2) is written over them that product has been issued.
#
# Per key tile, when the tile before and the tile after are there too (FWD_* statements):
#   max:   first half of the PV product (k-steps 0, 1)   | maximum of S(t)
#   exp_a: second half of the PV product (k-steps 2, 3)  | exponentials of scores 0..FWD_SPLIT-1
#   exp_b: S(t+1)                                        | exponentials of the other scores
# (an asm statement takes at most 30 operands, and the decision to move the running maximum sits
# between the first two). Workgroups of four wavefronts have twice the copies in the first one (max_4), and in stretches that
# need no masks a step of two statements, whose exponentials stay with the reference that there is:
#   free_pv: the whole PV product (16 MFMAs, 8 copies)   | exponentials of scores 0..FWD_FREE_SPLIT-1
#   free_qk: S(t+1)                                      | exponentials of the other scores
# Otherwise the same arithmetic and the same products as statements of
# their own (FWD_*_ONLY, FWD_QK, FWD_PV, FWD_PV_LATE), which give the same bits.
# ---------------------------------------------------------------------------
FWD_S = {"a": 112, "b": 144}
FWD_FIRST_PRIVATE = 112
FWD_RING0 = 176          # four fragment slots of four registers
FWD_LAST_PRIVATE = 191
FWD_SPLIT = 10
FWD_FREE_SPLIT = 16


def other(cur):
    return "b" if cur == "a" else "a"


def fwd_slot(slot):
    lo = FWD_RING0 + 4 * slot
    return lo, lo + 3


def fwd_acc(db):
    return "a[%d:%d]" % (16 * db, 16 * db + 15)


def weave(groups, valu, lead=0):
    """MFMA groups (wait, MFMA, the fragment reads behind it) with the vector instructions spread
    evenly behind them; `lead` of them go in front of the first group, under the first reads."""
    out = list(valu[:lead])
    rest = valu[lead:]
    pos = 0
    for gi, group in enumerate(groups):
        out += group
        want = (len(rest) * (gi + 1)) // len(groups)
        out += rest[pos:want]
        pos = want
    return out


def fwd_pf(cur, step):
    """P^T fragment of k-step `step` of the tile before the one in buffer `cur`."""
    lo = FWD_S[other(cur)] + 4 * step
    return "v[%d:%d]" % (lo, lo + 3)


def fwd_pv_groups(cur, steps):
    """MFMA groups of O^T[db] += V^T frag(step, db) * P^T[step] for the given k-steps; returns
    (head reads, groups). Operands by name: lo0-3, hi0-3, voff."""
    order = [(step, db) for step in steps for db in range(4)]
    n, ahead, slots = len(order), 4, 4

    def load(i):
        step, db = order[i]
        lo, _ = fwd_slot(i % slots)
        o = "%%[voff]+%d" % (step * 4096)
        return ["ds_read_b64_tr_b16 v[%d:%d], %%[lo%d] offset:%s" % (lo, lo + 1, db, o),
                "ds_read_b64_tr_b16 v[%d:%d], %%[hi%d] offset:%s" % (lo + 2, lo + 3, db, o)]

    head = ["s_waitcnt lgkmcnt(0)"]
    for i in range(min(ahead, n)):
        head += load(i)
    groups = []
    for i in range(n):
        later = min(ahead - 1, n - 1 - i)
        step, db = order[i]
        lo, hi = fwd_slot(i % slots)
        g = ["s_waitcnt lgkmcnt(%d)" % (2 * later),
             "v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], %s, %s" % (fwd_acc(db), lo, hi, fwd_pf(cur, step), fwd_acc(db))]
        if i + ahead < n:
            g += load(i + ahead)
        groups.append(g)
    return head, groups


def fwd_qk_groups(cur):
    """MFMA groups of S(t+1)^T = K Q^T into the buffer other than `cur`. Operands by name: rp0-7
    fragment pointers (k-step), q0-7 query fragments, koff."""
    nxt = FWD_S[other(cur)]
    n, ahead, slots = 16, 4, 4

    def load(i):
        ks, kb = divmod(i, 2)
        lo, hi = fwd_slot(i % slots)
        return ["ds_read_b128 v[%d:%d], %%[rp%d] offset:%%[koff]+%d" % (lo, hi, ks, kb * 8192)]

    head = ["s_waitcnt lgkmcnt(0)"]
    for i in range(ahead):
        head += load(i)
    groups = []
    for i in range(n):
        later = min(ahead - 1, n - 1 - i)
        ks, kb = divmod(i, 2)
        lo, hi = fwd_slot(i % slots)
        dst = "v[%d:%d]" % (nxt + 16 * kb, nxt + 16 * kb + 15)
        g = ["s_waitcnt lgkmcnt(%d)" % later,
             "v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], %%[q%d], %s" % (dst, lo, hi, ks, "0" if ks == 0 else dst)]
        if i + ahead < n:
            g += load(i + ahead)
        groups.append(g)
    return head, groups


def fwd_exp_ops(cur, lo, hi):
    """P = exp2(S c - m) in place for scores lo..hi-1 of buffer `cur` (lo, hi even), the running
    sum in score order, and the bf16 pairs; ordered so that nothing reads the result of the
    transcendental instruction directly in front of it. Operands: %[m] the reference, %[psum] the
    sum, %[c] log2 e (scalar)."""
    s0 = FWD_S[cur]
    ops = []
    for k in range(lo, hi + 2):
        if k < hi:
            ops.append("v_fma_f32 v%d, v%d, %%[c], -%%[m]" % (s0 + k, s0 + k))
        if lo <= k - 1 < hi:
            ops.append("v_exp_f32_e32 v%d, v%d" % (s0 + k - 1, s0 + k - 1))
        if lo <= k - 2 < hi:
            i = k - 2
            ops.append("v_add_f32_e32 %%[psum], %%[psum], v%d" % (s0 + i))
            if i % 2 == 1:
                ops.append("v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (s0 + i // 2, s0 + i - 1, s0 + i))
    return ops


def fwd_max_ops(cur):
    """%[mx] = log2 e times the maximum of the lane pair's scores in buffer `cur`; %[tmp] scratch."""
    s0 = FWD_S[cur]
    ops = ["v_max3_f32 %%[mx], v%d, v%d, v%d" % (s0, s0 + 1, s0 + 2)]
    for j in range(3, 31, 2):
        ops.append("v_max3_f32 %%[mx], %%[mx], v%d, v%d" % (s0 + j, s0 + j + 1))
    ops.append("v_max_f32_e32 %%[mx], %%[mx], v%d" % (s0 + 31))
    ops += ["v_mov_b32_e32 %[tmp], %[mx]", "s_nop 1", "v_permlane32_swap_b32 %[mx], %[tmp]",
            "v_max_f32_e32 %[mx], %[mx], %[tmp]", "v_mul_f32_e32 %[mx], %[c], %[mx]"]
    return ops


# Two wait states lie between a vector compare and the vector instruction that reads its bits: the bits of one are used
# behind the next two compares, and three scalar pairs take turns.
MASK_PAIRS = ("vcc", "s[96:97]", "s[98:99]")


def compare_and_use(compare, use):
    """One list of instructions per element: compare(e) and, two elements later, use(e); both give a mnemonic and its operands
    with {} where the pair stands."""
    def text(instruction, e):
        pair = MASK_PAIRS[e % 3]     # (vcc has the short encoding)
        return "%s_%s %s" % (instruction[0], "e32" if pair == "vcc" else "e64", instruction[1].format(pair))
    groups = [[text(compare(e), e)] + ([text(use(e - 2), e - 2)] if e >= 2 else []) for e in range(32)]
    groups[-1] += [text(use(e), e) for e in (30, 31)]
    return groups


def flatten(head, groups):
    return head + [ln for g in groups for ln in g]


def fwd_statements(cur):
    head_pv01, pv01 = fwd_pv_groups(cur, (0, 1))
    head_pv23, pv23 = fwd_pv_groups(cur, (2, 3))
    head_pv, pv = fwd_pv_groups(cur, (0, 1, 2, 3))
    head_qk, qk = fwd_qk_groups(cur)
    key_offset = lambda i: 32 * (i // 16) + 8 * ((i % 16) // 4) + (i % 16) % 4
    s0 = FWD_S[cur]
    select = lambda i: ("v_cndmask_b32", "v%d, %%[ninf], v%d, {}" % (s0 + i, s0 + i))
    causal = flatten([], compare_and_use(lambda i: ("v_cmp_le_i32", "{}, %d, %%[rel]" % key_offset(i)), select))
    # ids: the tile's 64 key ids sit in LDS in key order; %[idp] is this lane's address of key
    # 4 * (lane / 32), so the quad of registers 4 q .. 4 q + 3 of block kb is the 16 bytes at
    # offset 4 * (32 kb + 8 q). Quads go through the fragment ring (four in flight).
    ids = ["s_waitcnt lgkmcnt(0)"]
    quad_regs = lambda q: FWD_RING0 + 4 * (q % 4)
    quad_read = lambda q: "ds_read_b128 v[%d:%d], %%[idp] offset:%d" % (
        quad_regs(q), quad_regs(q) + 3, 4 * (32 * (q // 4) + 8 * (q % 4)))
    ids += [quad_read(q) for q in range(4)]
    by_id = compare_and_use(lambda i: ("v_cmp_eq_u32", "{}, %%[segq], v%d" % (quad_regs(i // 4) + i % 4)), select)
    for q in range(8):
        ids.append("s_waitcnt lgkmcnt(%d)" % min(3, 7 - q))
        ids += flatten([], by_id[4 * q:4 * q + 4])
        if q + 4 < 8:
            ids.append(quad_read(q + 4))
    return {
        # the three interleaved statements
        "MAX": head_pv01 + weave(fwd_with_copies(pv01, 2), fwd_max_ops(cur)),
        # with twice the copies, for workgroups of four wavefronts
        "MAX_4": head_pv01 + weave(fwd_with_copies(pv01, 4), fwd_max_ops(cur)),
        # the step in two statements, without the maximum: the exponentials against the reference as it is
        "FREE_PV": head_pv + weave(fwd_with_copies(pv, 4), fwd_exp_ops(cur, 0, FWD_FREE_SPLIT)),
        "FREE_QK": head_qk + weave(qk, fwd_exp_ops(cur, FWD_FREE_SPLIT, 32), lead=6) + TAIL,
        "EXP_A": head_pv23 + weave(pv23, fwd_exp_ops(cur, 0, FWD_SPLIT)),
        "EXP_B": head_qk + weave(qk, fwd_exp_ops(cur, FWD_SPLIT, 32), lead=6) + TAIL,
        # the same pieces on their own
        "MAX_ONLY": fwd_max_ops(cur),
        "EXP_ONLY": fwd_exp_ops(cur, 0, 32),
        "PV": flatten(head_pv, pv) + TAIL,
        "PV_LATE": flatten(head_pv23, pv23) + TAIL,
        "QK": flatten(head_qk, qk) + TAIL,
        # the first scores of a query tile, with the clearing of the output accumulator behind the MFMAs
        "QK_ZERO": head_qk + weave(qk, fwd_accumulator_statements()["ZERO"]) + TAIL,
        # masks: scores of pairs that are not allowed become -inf. CAUSAL: allowed = key offset in the
        # tile <= %[rel] (per lane)
        "MASK_CAUSAL": causal,
        # IDS: the key's id (read here from the id ring in LDS) differs from %[segq] (per lane)
        "MASK_IDS": ids,
    }


def fwd_with_copies(groups, passes):
    """The step's global -> LDS copies of this wavefront (V rows of this tile, then K rows of the
    tile after next: `passes` pieces of 1 KB each) placed behind the MFMAs: their issue then costs
    the matrix pipe nothing. Copy g: m0 = %[d<g>] (LDS destination, scalar), source = scalar base
    %[vsrc] (g < passes) or %[ksrc] plus the lane's byte offset %[off<g % passes>]. m0 is set one
    MFMA ahead of its copy; the last copy closes the statement."""
    out = [list(g) for g in groups]
    n = 2 * passes
    assert n <= len(groups)
    for g in range(n):
        load = "global_load_lds_dwordx4 %%[off%d], %%[%s]" % (g % passes, "vsrc" if g < passes else "ksrc")
        out[g].append("s_mov_b32 m0, %%[d%d]" % g)
        if g + 1 < len(groups):
            out[g + 1] = out[g + 1][:2] + [load] + out[g + 1][2:]
        else:
            out.append([load])
    return out


def fwd_accumulator_statements():
    """The output accumulator O^T (128 x 32 queries) lives in a[0:63], which only these statements
    and the PV products name. ZERO; SCALE: every element times %[alpha] (per lane: the row's
    factor), eight elements in flight through the fragment ring; the read-out uses CT_DKVW_READ."""
    zero = ["v_accvgpr_write_b32 a%d, 0" % r for r in range(64)]
    scale = []
    ring = list(range(FWD_RING0, FWD_RING0 + 8))
    for base in range(0, 64, 8):
        scale += ["v_accvgpr_read_b32 v%d, a%d" % (ring[e], base + e) for e in range(8)]
        scale += ["v_mul_f32_e32 v%d, %%[alpha], v%d" % (ring[e], ring[e]) for e in range(8)]
        scale += ["v_accvgpr_write_b32 a%d, v%d" % (base + e, ring[e]) for e in range(8)]
    return {"ZERO": zero, "SCALE": scale + ["s_nop 1"]}


def fwd_private_clobbers():
    return ", ".join(['"v%d"' % r for r in range(FWD_FIRST_PRIVATE, FWD_LAST_PRIVATE + 1)] +
                     ['"a%d"' % r for r in range(64)])


class Stream:
    """Instruction list with in-order tracking of the LDS reads in flight (lgkmcnt)."""

    def __init__(self, head=("s_waitcnt lgkmcnt(0)",)):
        self.lines = list(head)
        self.pending = []

    def lds(self, text, tag):
        self.lines.append(text)
        self.pending.append(tag)
        assert len(self.pending) <= 15, "lgkmcnt holds at most 15"

    def wait(self, tag):
        if tag not in self.pending:
            return
        i = len(self.pending) - 1 - self.pending[::-1].index(tag)
        self.lines.append("s_waitcnt lgkmcnt(%d)" % (len(self.pending) - 1 - i))
        self.pending = self.pending[i + 1:]

    def wait_all(self):
        self.lines.append("s_waitcnt lgkmcnt(0)")
        self.pending = []

    def emit(self, text):
        self.lines.append(text)


def w_acc(i):
    """Accumulator i of the wide kernel: 0-3 dV of key block 0 (column block db), 4-7 dV of key
    block 1, 8-11 dK of key block 0, 12-15 dK of key block 1. They live in fixed accumulation
    registers for the whole kernel and are never handed to the compiler."""
    return "a[%d:%d]" % (16 * i, 16 * i + 15)


# dK/dV, a step as one stream: S first, then dP with the exponents of S behind its
# MFMAs, then dV with the dS arithmetic behind its MFMAs, then dK. Fixed registers (declared as clobbers): a bit
# per pair that is allowed, the bf16 P fragments, the address of a V fragment, S, dP (its first 8 registers later hold the bf16 dS fragments) and the ring; the
# sums are a[0:127] for the whole kernel (w_acc: 0-3 dV, 4-7 dK) and never handed to the compiler, so a step does not end
# with the wait states behind its last MFMA (1.5 % of the kernel): whoever reads the sums waits. Between its streams a
# wavefront issues behind the other one of its SIMD (the other way round 0.5 to 1 % longer). The matrix pipe is busy 64 % of
# the time with five fragment slots, 61.5 as two sequences (products, sums) with the arithmetic between them ([2, 8192, 16/16] whole
# rows); [4, 4096, 32/8] documents of 64 to 4096 682 -> 642 us, [2, 8192, 16/16] of 64 to 2000 235 -> 224. Five slots instead
# of six 0.2 % longer, seven 0.5 % shorter in launches of one round and 0.7 % longer in large ones.
DKVS_SLOTS = 6
DKVS_RING0 = 128 - 4 * DKVS_SLOTS
DKVS_DP = DKVS_RING0 - 16
DKVS_S = DKVS_DP - 16
DKVS_ADDR = DKVS_S - 1
DKVS_ALLOWED = DKVS_ADDR - 1
DKVS_P = DKVS_ALLOWED - 8   # (register runs begin at even numbers)


def dkv_step_sequence(mask, stores):
    """operands: %0-%7 K fragments, %8-%15 row-fragment pointers, %16-%19 transposed fragments, lo, and %20-%23, hi, %24
    pointer of this lane's statistics (LDS base + 16 * (lane / 32)), %25 scale * log2(e) and %26 byte offset of this
    wavefront's V rows (scalar), %27 byte offset of the stage (Q tile, dO tile 8192 later, -lse / scale at 16384, -delta at
    16512). With `mask` some pair is not allowed, and its sum becomes %28 (scalar): those with another id than %29 among the
    ids of the query rows (at 16640 of the stage), and with "ends" those whose key %30 lies behind the row's visible end
    (at 16768), with "rows" those where %30, the key less the number of the half's first row, is more than the row's own. With `stores` the dS block leaves as well: behind those its address (scalar pair)
    and 16 * lane.

    Scalar loads may be in flight where the stream begins: its first wait is for everything, and no other counts them.
    """
    st = Stream(head=[])
    stage = "%27"
    block = lambda base: "v[%d:%d]" % (base, base + 15)

    def stats(base, offset):
        for qd in range(4):
            st.lds("ds_read_b128 v[%d:%d], %%24 offset:%s+%d" % (base + 4 * qd, base + 4 * qd + 3, stage, offset + 32 * qd), "stat")

    def slot(r):
        lo = DKVS_RING0 + 4 * (r % DKVS_SLOTS)
        return lo, "v[%d:%d]" % (lo, lo + 3)

    reads, mfmas = [], []
    for ks in range(8):
        reads.append(["ds_read_b128 {v4}, %%%d offset:%s" % (8 + ks, stage)])
        mfmas.append(("v_mfma_f32_32x32x16_bf16 %s, {r0}, %%%d, %s" % (block(DKVS_S), ks, block(DKVS_S)), [ks]))
    for ks in range(8):
        base = len(reads)
        reads.append(["ds_read_b128 {v4}, %%%d offset:%s+8192" % (8 + ks, stage)])
        reads.append(["v_add_u32_e32 v%d, %%26, %%%d" % (DKVS_ADDR, 8 + ks), "ds_read_b128 {v4}, v%d" % DKVS_ADDR])
        mfmas.append(("v_mfma_f32_32x32x16_bf16 %s, {r0}, {r1}, %s" % (block(DKVS_DP), block(DKVS_DP)), [base, base + 1]))
    for which, source in ((0, DKVS_P), (1, DKVS_DP)):   # dV (P^T, dO), dK (dS^T, Q)
        for step in range(2):
            for db in range(4):
                off = "%s+%d" % (stage, step * 4096 + (8192 if which == 0 else 0))
                reads.append(["ds_read_b64_tr_b16 {v2lo}, %%%d offset:%s" % (16 + db, off),
                              "ds_read_b64_tr_b16 {v2hi}, %%%d offset:%s" % (20 + db, off)])
                a = w_acc(4 * which + db)
                mfmas.append(("v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], {r0}, %s" % (a, source + 4 * step, source + 4 * step + 3, a),
                              [len(reads) - 1]))

    # A product's sums are read two MFMAs after its last one at the earliest: they have left the matrix pipe by then.
    fill = [[] for _ in range(len(mfmas) + 1)]
    packed_at = {}
    for e in range(16):
        t = 9 + (e * 9) // 16
        if mask:   # (the address register is free between the pairs of instructions that use it)
            fill[t] += ["v_bfe_i32 v%d, v%d, %d, 1" % (DKVS_ADDR, DKVS_ALLOWED, 15 - e),
                        "v_bfi_b32 v%d, v%d, v%d, %%28" % (DKVS_S + e, DKVS_ADDR, DKVS_S + e)]
        fill[t] += ["v_mul_f32_e32 v%d, %%25, v%d" % (DKVS_S + e, DKVS_S + e), "v_exp_f32_e32 v%d, v%d" % (DKVS_S + e, DKVS_S + e)]
        t_ds = 17 + (e * 9) // 16
        fill[t_ds] += ["v_mul_f32_e32 v%d, v%d, v%d" % (DKVS_DP + e, DKVS_S + e, DKVS_DP + e)]
        if e % 2 == 1:
            k = e // 2
            fill[t + 1] += ["v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (DKVS_P + k, DKVS_S + 2 * k, DKVS_S + 2 * k + 1)]
            fill[t_ds] += ["v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (DKVS_DP + k, DKVS_DP + 2 * k, DKVS_DP + 2 * k + 1)]
            packed_at[e] = (t + 1, t_ds)
    assert packed_at[7][0] < 16 and packed_at[15][0] < 20 and packed_at[7][1] < 24 and packed_at[15][1] < 28
    if stores:
        address, lane = ("%31", "%32") if mask else ("%28", "%29")
        for half, e in ((0, 7), (1, 15)):
            fill[packed_at[e][1] + 2] += ["global_store_dwordx4 %s, v[%d:%d], %s offset:%d" % (
                lane, DKVS_DP + 4 * half, DKVS_DP + 4 * half + 3, address, 1024 * half)]

    # The bits of the pairs, four rows at a time behind two MFMAs of S: ids and ends go where the P fragments will be.
    def mask_reads(qd):
        st.lds("ds_read_b128 v[%d:%d], %%24 offset:%s+%d" % (DKVS_P, DKVS_P + 3, stage, 16640 + 32 * qd), "mask")
        if mask == "ends":
            st.lds("ds_read_b128 v[%d:%d], %%24 offset:%s+%d" % (DKVS_P + 4, DKVS_P + 7, stage, 16768 + 32 * qd), "mask")

    def mask_bits(qd, e):
        limit = "v_cmp_le_i32_e64 s[96:97], %%30, v%d" % (DKVS_P + 4 + e) if mask == "ends" else "v_cmp_ge_i32_e64 s[96:97], %d, %%30" % (8 * qd + e)
        return ["v_cmp_eq_u32_e32 vcc, %%29, v%d" % (DKVS_P + e), limit, "s_and_b64 vcc, vcc, s[96:97]",
                "v_addc_co_u32_e32 v%d, vcc, v%d, v%d, vcc" % (DKVS_ALLOWED, DKVS_ALLOWED, DKVS_ALLOWED)]

    state = {"issued": 0}
    consumed = [False] * len(reads)

    def issue_reads():
        while state["issued"] < len(reads):
            r = state["issued"]
            if r >= DKVS_SLOTS and not consumed[r - DKVS_SLOTS]:
                break
            lo, v4 = slot(r)
            for text in reads[r]:
                text = text.format(v4=v4, v2lo="v[%d:%d]" % (lo, lo + 1), v2hi="v[%d:%d]" % (lo + 2, lo + 3))
                (st.lds(text, r) if text.startswith("ds_") else st.emit(text))
            state["issued"] += 1

    stats(DKVS_S, 16384)
    issue_reads()
    st.wait_all()
    st.emit("s_setprio 1")
    if mask:
        st.emit("v_mov_b32_e32 v%d, 0" % DKVS_ALLOWED)
    for i, (text, needs) in enumerate(mfmas):
        st.wait(needs[-1])
        st.emit(text.format(**{"r%d" % n: slot(r)[1] for n, r in enumerate(needs)}))
        for r in needs:
            consumed[r] = True
        if i == 0:
            stats(DKVS_DP, 16512)
        if mask and i < 8:
            if i % 2 == 0:
                mask_reads(i // 2)
            else:
                st.wait("mask")
                for e in range(4):
                    for line in mask_bits(i // 2, e):
                        st.emit(line)
        issue_reads()
        for line in fill[i]:
            st.emit(line)
    assert not fill[len(mfmas)] and state["issued"] == len(reads)
    return st.lines + ["s_setprio 0"]


# dQ, a key tile of 64 keys as one stream: S and dP of its first half, S of the second with the first half's dS behind its
# MFMAs, dP of the second, the first half's share of dQ with the second's dS behind it, the second's share. Fixed registers
# (declared as clobbers): one temporary, three score blocks (S0, later dP1; dP0; S1; the first 8 registers of a dP block
# later hold its bf16 dS fragments) and the fragment ring; the sums are a[0:63] for the whole query tile. (With the two
# halves one after the other, each as two sequences with the arithmetic between them: [2, 8192, 16/16], documents of 64 to
# 2000, the kernel 191 us, now 178; [2, 10496, 64/8] of 248 to 3277 1214 and 1095; whole rows of 16384, 8/1, 769 and 703;
# [1, 6144, 4/4] of 100 to 600 38.3 and 31.9. Five or seven fragment slots and a raised issue priority, as in dK/dV, change nothing.)
DQS_SLOTS = 6
DQS_RING0 = 192 - 4 * DQS_SLOTS
DQS_S = (DQS_RING0 - 48, DQS_RING0 - 16)
DQS_DP = (DQS_RING0 - 32, DQS_RING0 - 48)
DQS_TMP = DQS_RING0 - 49
DQS_FIRST = DQS_TMP


def dq_step_sequence(masked):
    """operands: %0-%7 Q and %8-%15 dO fragments, %16-%23 row-fragment pointers, %24-%27 transposed fragments, lo, and
    %28-%31, hi, %32 lse * log2(e), %33 delta of the lane's query row, %34 log2(e) (scalar), %35 byte offset of the stage (64 K
    rows, 64 V rows 16384 later). With `masked` bit e of %36 tells whether the pair of element e (second half: 16 + e) is
    allowed, and the score of one that is not becomes %37 (scalar).

    Scalar loads may be in flight where the stream begins: its first wait is for everything, and no other counts them.
    """
    st = Stream(head=[])
    stage = "%35"
    block = lambda base: "v[%d:%d]" % (base, base + 15)

    def slot(r):
        lo = DQS_RING0 + 4 * (r % DQS_SLOTS)
        return lo, "v[%d:%d]" % (lo, lo + 3)

    reads, mfmas = [], []
    for half in range(2):
        for which, base in ((0, DQS_S[half]), (1, DQS_DP[half])):
            for ks in range(8):
                reads.append(["ds_read_b128 {v4}, %%%d offset:%s+%d" % (16 + ks, stage, 16384 * which + 8192 * half)])
                mfmas.append("v_mfma_f32_32x32x16_bf16 %s, {r0}, %%%d, %s" % (block(base), 8 * which + ks, block(base) if ks else "0"))
    for half in range(2):
        for step in range(2):
            for db in range(4):
                off = "%s+%d" % (stage, 8192 * half + 4096 * step)
                reads.append(["ds_read_b64_tr_b16 {v2lo}, %%%d offset:%s" % (24 + db, off),
                              "ds_read_b64_tr_b16 {v2hi}, %%%d offset:%s" % (28 + db, off)])
                source = DQS_DP[half] + 4 * step
                mfmas.append("v_mfma_f32_32x32x16_bf16 %s, {r0}, v[%d:%d], %s" % (w_acc(db), source, source + 3, w_acc(db)))

    # A product's scores are read two MFMAs after its last one at the earliest: they have left the matrix pipe by then.
    fill = [[] for _ in mfmas]
    for half in range(2):
        S, DP = DQS_S[half], DQS_DP[half]
        for e in range(16):
            t = 9 + 16 * half + (e * 7) // 16
            # (the last pair is packed behind MFMA 42 and read by MFMA 44: what lies between are the two wait states that it takes)
            t_ds = 17 + (e * 7) // 16 if half == 0 else 33 + (e * 10) // 16
            if masked:
                fill[t] += ["v_bfe_i32 v%d, %%36, %d, 1" % (DQS_TMP, 16 * half + e),
                            "v_bfi_b32 v%d, v%d, v%d, %%37" % (S + e, DQS_TMP, S + e)]
            fill[t] += ["v_fma_f32 v%d, v%d, %%34, -%%32" % (S + e, S + e), "v_exp_f32_e32 v%d, v%d" % (S + e, S + e)]
            fill[t_ds] += ["v_sub_f32_e32 v%d, v%d, %%33" % (DP + e, DP + e), "v_mul_f32_e32 v%d, v%d, v%d" % (DP + e, S + e, DP + e)]
            if e % 2 == 1:
                k = e // 2
                fill[t_ds] += ["v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (DP + k, DP + 2 * k, DP + 2 * k + 1)]

    state = {"issued": 0, "consumed": 0}

    def issue_reads():
        while state["issued"] < min(len(reads), state["consumed"] + DQS_SLOTS):
            r = state["issued"]
            lo, v4 = slot(r)
            for text in reads[r]:
                st.lds(text.format(v4=v4, v2lo="v[%d:%d]" % (lo, lo + 1), v2hi="v[%d:%d]" % (lo + 2, lo + 3)), r)
            state["issued"] += 1

    issue_reads()
    st.wait_all()
    for i, text in enumerate(mfmas):
        st.wait(i)
        st.emit(text.format(r0=slot(i)[1]))
        state["consumed"] += 1
        issue_reads()
        for line in fill[i]:
            st.emit(line)
    return st.lines


def dq_ids_sequence():
    """%0: bit e tells whether the id of element e's key is %2 (elements as in the stream above); %1 pointer of the lane's ids
    (LDS address of the ids + 16 * (lane / 32)), %3 byte offset of the stage."""
    lines = ["s_waitcnt lgkmcnt(0)"]
    base = DQS_DP[1]
    for q in range(8):
        lines.append("ds_read_b128 v[%d:%d], %%1 offset:%%3+%d" % (base + 4 * q, base + 4 * q + 3, 32 * (7 - q)))
    lines.append("v_mov_b32_e32 %0, 0")
    # (the last element first; what a carry leaves in its pair nothing reads)
    bits = compare_and_use(lambda i: ("v_cmp_eq_u32", "{}, %%2, v%d" % (base + (i | 3) - i % 4)),
                           lambda i: ("v_addc_co_u32", "%0, {0}, %0, %0, {0}"))
    for q in range(8):
        lines.append("s_waitcnt lgkmcnt(%d)" % (7 - q))
        lines += flatten([], bits[4 * q:4 * q + 4])
    return lines


# ---------------------------------------------------------------------------
# dK/dV, wide form: one wavefront per SIMD owns 64 keys (two 32-key blocks) and runs a whole
# (head, query block) step as one instruction stream. With nothing else resident on the SIMD the
# wavefront's exponent / dS arithmetic has to sit between its own MFMAs: the arithmetic of key
# block 0 is placed under the S / dP MFMAs of key block 1, that of key block 1 under the dV / dK
# MFMAs of key block 0.
#
# Fixed registers (declared as clobbers): a ring of 5 fragment slots, the score / dP blocks of
# both key blocks (their first 8 registers later hold the bf16 P and dS fragments) and the 16
# lse2 / delta values of this lane's query rows.
# ---------------------------------------------------------------------------
W_SLOTS = 5
W_RING0 = 256 - 4 * W_SLOTS
W_S = (W_RING0 - 64, W_RING0 - 32)      # S^T accumulators of key block 0 / 1 (16 registers each)
W_DP = (W_RING0 - 48, W_RING0 - 16)     # dP accumulators
W_ADDR = W_RING0 - 65                   # address of a V fragment
W_FIRST = W_ADDR


class WideOperands:
    """Names of the asm operands of one stream (strings such as "%12")."""

    def __init__(self, first_input, masked):
        n = first_input
        self.k = [["%%%d" % (n + 8 * kb + ks) for ks in range(8)] for kb in range(2)]   # K fragments [kb][ks]
        self.rp = ["%%%d" % (n + 16 + ks) for ks in range(8)]                          # row-fragment pointers
        self.tlo = ["%%%d" % (n + 24 + db) for db in range(4)]                         # transposed fragments, lo
        self.thi = ["%%%d" % (n + 28 + db) for db in range(4)]                         # ... hi
        self.stat = "%%%d" % (n + 32)      # pointer of this lane's statistics (LDS base + 16 * (lane / 32))
        self.scale = "%%%d" % (n + 33)     # scale * log2(e), scalar
        self.voff = "%%%d" % (n + 34)      # byte offset of this wavefront's V rows, scalar
        self.src = ["%%%d" % (n + 35 + i) for i in range(4)]   # Q rows, dO rows, two statistics arrays (scalar pairs)
        self.tile_base = "%%%d" % (n + 39)  # LDS address of this wavefront's first slot of a Q tile at stage offset 0
        self.stat_base = "%%%d" % (n + 40)  # LDS address of its first statistics array at stage offset 0
        self.count = n + 41
        if masked:
            self.sinit = ["%%%d" % (n + 41), "%%%d" % (n + 42)]
            self.count = n + 43


def dkvw_stream(o, stage, other, loff, lane16, masked=False):
    """One (head, query block) step of the wide dK/dV kernel for both key blocks.

    `stage` / `other`: byte offsets (operand names or numbers) of the stage that is read (Q tile, dO
    tile 8192 later, -lse / scale at 16384, -delta at 16512) and of the stage the next item is
    copied into; `loff` the four registers with this thread's source offsets of a 32 x 128 tile,
    `lane16` the register with 16 * lane.

    The copies of the next item (its Q and dO rows and statistics) are issued from inside the
    stream, one behind each of the first ten MFMAs.

    The S blocks start from -lse / scale of their query rows (read from the stage) and the dP
    blocks from -delta. With `masked`, the starting values of the two S blocks come in registers
    instead (o.sinit): the caller has put -inf where a pair is not allowed, and the sum, the
    probability and dS of such a pair are then -inf, 0 and 0 without any instruction here knowing
    about masks.
    """
    st = Stream()

    def stats(kb):
        # The S and dP blocks start from the per-row terms instead of 0: -lse / scale and -delta of
        # the block's 16 query rows (4 consecutive rows per read, the accumulator's own order).
        for qd in range(0 if masked else 4):
            st.lds("ds_read_b128 v[%d:%d], %s offset:%s+%d" % (W_S[kb] + 4 * qd, W_S[kb] + 4 * qd + 3, o.stat, stage,
                                                                16384 + 32 * qd), "stat%d" % kb)
        for qd in range(4):
            st.lds("ds_read_b128 v[%d:%d], %s offset:%s+%d" % (W_DP[kb] + 4 * qd, W_DP[kb] + 4 * qd + 3, o.stat, stage,
                                                                16512 + 32 * qd), "stat%d" % kb)

    stats(0)

    def acc16(base):
        return "v[%d:%d]" % (base, base + 15)

    def slot(r):
        lo = W_RING0 + 4 * (r % W_SLOTS)
        return lo, "v[%d:%d]" % (lo, lo + 3)

    # ---- the reads (in issue order) and the MFMAs (in issue order, each naming the reads it needs)
    reads, mfmas = [], []
    for kb in range(2):
        for ks in range(8):
            base = len(reads)
            reads.append(["ds_read_b128 {v4}, %s offset:%s" % (o.rp[ks], stage)])                   # Q
            reads.append(["ds_read_b128 {v4}, %s offset:%s+8192" % (o.rp[ks], stage)])              # dO
            reads.append(["v_add_u32_e32 v%d, %s, %s" % (W_ADDR, o.voff, o.rp[ks]),                  # V
                          "ds_read_b128 {v4}, v%d offset:%d" % (W_ADDR, 8192 * kb)])
            c_s = o.sinit[kb] if (masked and ks == 0) else acc16(W_S[kb])
            mfmas.append(("v_mfma_f32_32x32x16_bf16 %s, {r0}, %s, %s" % (acc16(W_S[kb]), o.k[kb][ks], c_s), [base]))
            mfmas.append(("v_mfma_f32_32x32x16_bf16 %s, {r0}, {r1}, %s" % (acc16(W_DP[kb]), acc16(W_DP[kb])), [base + 1, base + 2]))
    for kb in range(2):
        for step in range(2):
            for db in range(4):
                for which in range(2):  # 0: dV (P^T, dO), 1: dK (dS^T, Q)
                    off = "%s+%d" % (stage, step * 4096 + (8192 if which == 0 else 0))
                    reads.append(["ds_read_b64_tr_b16 {v2lo}, %s offset:%s" % (o.tlo[db], off),
                                  "ds_read_b64_tr_b16 {v2hi}, %s offset:%s" % (o.thi[db], off)])
                    acc = w_acc((0 if which == 0 else 8) + 4 * kb + db)
                    src = (W_S if which == 0 else W_DP)[kb] + 4 * step
                    mfmas.append(("v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], {r0}, %s" % (acc, src, src + 3, acc),
                                  [len(reads) - 1]))
    assert len(mfmas) == 64

    # ---- the arithmetic, attached to MFMA slots. Element e of key block kb starts under MFMA
    # 16 + 16 kb + 11 e / 8: elements 0-7 are packed before the block's first dV / dK MFMA (32 + 16
    # kb) needs them, elements 8-15 before its ninth does, and no MFMA has much more than one
    # element behind it.
    fill = [[] for _ in range(len(mfmas) + 1)]
    for kb in range(2):
        S, DP = W_S[kb], W_DP[kb]
        done = {}
        for e in range(16):
            t = 16 + 16 * kb + (11 * e) // 8
            fill[t] += ["v_mul_f32_e32 v%d, %s, v%d" % (S + e, o.scale, S + e),
                        "v_exp_f32_e32 v%d, v%d" % (S + e, S + e)]
            # the dP block is first read two MFMAs later: its last MFMA has long retired by then
            fill[t + 2] += ["v_mul_f32_e32 v%d, v%d, v%d" % (DP + e, S + e, DP + e)]
            done[e] = t + 2
            if e % 2 == 1:
                k = e // 2
                fill[t + 2] += ["v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (S + k, S + 2 * k, S + 2 * k + 1),
                                "v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (DP + k, DP + 2 * k, DP + 2 * k + 1)]
        assert done[7] < 32 + 16 * kb and done[15] < 40 + 16 * kb

    # ---- emission: reads run ahead of their MFMAs as far as the ring allows
    state = {"issued": 0}
    consumed = [False] * len(reads)

    def issue_reads():
        while state["issued"] < len(reads):
            r = state["issued"]
            if r >= W_SLOTS and not consumed[r - W_SLOTS]:
                break
            lo, v4 = slot(r)
            for text in reads[r]:
                text = text.format(v4=v4, v2lo="v[%d:%d]" % (lo, lo + 1), v2hi="v[%d:%d]" % (lo + 2, lo + 3))
                if text.startswith("ds_"):
                    st.lds(text, r)
                else:
                    st.emit(text)
            state["issued"] += 1

    # the copies: (instructions in front of the MFMA, instructions behind it)
    copies = []
    for which in range(2):
        for n in range(4):
            copies.append((["s_add_u32 m0, %s, %s+%d" % (o.tile_base, other, 8192 * which + 2048 * n)],
                           ["global_load_lds_dwordx4 %s, %s" % (loff[n], o.src[which])]))
    for which in range(2):
        copies.append((["s_add_u32 m0, %s, %s+%d" % (o.stat_base, other, 128 * which)],
                       ["s_mov_b64 exec, 0xff", "global_load_lds_dwordx4 %s, %s" % (lane16, o.src[2 + which]),
                        "s_mov_b64 exec, -1"]))

    issue_reads()
    for i, (text, needs) in enumerate(mfmas):
        st.wait(needs[-1])
        if i < len(copies):
            for line in copies[i][0]:
                st.emit(line)
        names = {"r%d" % n: slot(r)[1] for n, r in enumerate(needs)}
        st.emit(text.format(**names))
        if i < len(copies):
            for line in copies[i][1]:
                st.emit(line)
        for r in needs:
            consumed[r] = True
        if i == 3:
            stats(1)   # (the registers are free: their last readers were the previous step's MFMAs)
        issue_reads()
        for line in fill[i]:
            st.emit(line)
    assert not fill[64] and state["issued"] == len(reads)
    return st.lines


def dkvw_step_sequence(masked=False):
    """A single step. operands: %0-%40 as WideOperands(0) lays them out, %41 / %42 the S starting
    values (masked form only), then the stage offset, the other stage's offset (immediates), the four
    source offsets of this thread and 16 * lane."""
    o = WideOperands(0, masked)
    n = o.count
    stage, other = "%%%d" % n, "%%%d" % (n + 1)
    loff = ["%%%d" % (n + 2 + i) for i in range(4)]
    return dkvw_stream(o, stage, other, loff, "%%%d" % (n + 6), masked) + TAIL


def dkvw_run_sequence():
    """A run of all-allowed steps over consecutive query blocks of one head: the stream of the
    stage the run starts on, then the stream of the other stage, and so on, each followed by the
    wait for the copies it issued and the workgroup barrier; the source offsets advance by one
    query block per step.

    operands: %0 steps left (scalar, counted down to 0); %1-%4 this thread's source offsets and %5
    16 * lane (advanced); %6-%46 as WideOperands(6) lays them out; %47 bytes between the Q rows of
    consecutive query blocks (scalar); %48 / %49 byte offsets of the stage the run starts on and of
    the other one.
    """
    o = WideOperands(6, False)
    assert o.count == 47
    loff, lane16 = ["%1", "%2", "%3", "%4"], "%5"
    close = ["s_waitcnt vmcnt(0)", "s_barrier"] + ["v_add_u32_e32 %s, %%47, %s" % (r, r) for r in loff] + [
        "v_add_u32_e32 %s, 0x80, %s" % (lane16, lane16), "s_sub_u32 %0, %0, 1", "s_cmp_eq_u32 %0, 0"]
    lines = ["dkvw_run_%=:"]
    lines += dkvw_stream(o, "%48", "%49", loff, lane16) + close + ["s_cbranch_scc1 dkvw_run_end_%="]
    lines += dkvw_stream(o, "%49", "%48", loff, lane16) + close + ["s_cbranch_scc0 dkvw_run_%="]
    lines += ["dkvw_run_end_%=:"]
    return lines + TAIL


def accumulators_zero(registers):
    return ["v_accvgpr_write_b32 a%d, 0" % r for r in range(registers)]


def dkvw_read():
    """operands: %0-%15 the 16 values of one accumulator, %16 its first register number."""
    return ["v_accvgpr_read_b32 %%%d, a[%%16+%d]" % (e, e) for e in range(16)]


def clobbers():
    regs = ", ".join('"v%d"' % r for r in range(SCRATCH0, SCRATCH0 + 16))
    dq = ", ".join('"v%d"' % r for r in range(DQS_FIRST, 192))
    dq_accs = ", ".join('"a%d"' % r for r in range(64))
    step = ", ".join('"v%d"' % r for r in range(DKVS_P, 128))
    step_accs = ", ".join('"a%d"' % r for r in range(128))
    wide = ", ".join('"v%d"' % r for r in range(W_FIRST, 256))
    accs = ", ".join('"a%d"' % r for r in range(256))
    pairs = '"vcc", "s96", "s97", "s98", "s99"'
    return ("#define CT_MASK_PAIRS %s\n\n#define CT_ATTN_ASM_SCRATCH %s\n\n#define CT_DQ_STEP_SCRATCH %s\n\n#define CT_DQ_ACCUMULATORS %s\n\n"
            "#define CT_DKV_STEP_SCRATCH %s\n\n"
            "#define CT_DKV_ACCUMULATORS %s\n\n"
            "#define CT_DKVW_ASM_SCRATCH %s\n\n"
            "#define CT_DKVW_ACCUMULATORS %s\n\n#define CT_FWD_PRIVATE %s\n" % (pairs, regs, dq, dq_accs, step, step_accs, wide, accs,
                                                                             fwd_private_clobbers()))


if __name__ == "__main__":
    print("// Generated by gen_attn_asm.py -- do not edit by hand.")
    print(emit(pv_sequence(4, 4), "CT_ATTN_PV_SEQUENCE"))
    print(emit(qk_sequence(4, 4), "CT_ATTN_QK_SEQUENCE"))
    for cur in ("a", "b"):
        for name, lines in fwd_statements(cur).items():
            print(emit(lines, "CT_FWD_%s_%s" % (name, cur.upper())))
    for name, lines in fwd_accumulator_statements().items():
        print(emit(lines, "CT_FWD_ACC_%s" % name))
    print(emit(dq_step_sequence(False), "CT_DQ_STEP_SEQUENCE"))
    print(emit(dq_step_sequence(True), "CT_DQ_STEP_MASKED_SEQUENCE"))
    print(emit(dq_ids_sequence(), "CT_DQ_IDS_SEQUENCE"))
    print(emit(accumulators_zero(64), "CT_DQ_ZERO"))
    for mask in ("", "ends", "rows"):
        for stores in (False, True):
            print(emit(dkv_step_sequence(mask, stores), "CT_DKV_STEP_%s%sSEQUENCE" % (mask.upper() + "_" * bool(mask), "STORE_" * stores)))
    print(emit(accumulators_zero(128), "CT_DKV_ZERO"))
    print(emit(dkvw_step_sequence(), "CT_DKVW_FAST_SEQUENCE"))
    print(emit(dkvw_step_sequence(masked=True), "CT_DKVW_MASKED_SEQUENCE"))
    print(emit(dkvw_run_sequence(), "CT_DKVW_RUN_SEQUENCE"))
    print(emit(accumulators_zero(256), "CT_DKVW_ZERO"))
    print(emit(dkvw_read(), "CT_DKVW_READ"))
    print(clobbers())
