"""Generates ct_gemm_asm.inc: the hand-scheduled main loops of the 256 x 256 and 128 x 128 GEMM tiles.

One wavefront runs on each SIMD, so whatever the wavefront issues between two MFMAs must fit
into the 32 cycles the matrix pipe is busy with the first of them, or the pipe drains. A
global -> LDS copy costs about 23 cycles to issue and an LDS fragment read 4 to 8; issued in
bursts (as the compiler schedules them) they stall the MFMA stream for hundreds of cycles per
k-step. The sequence below fixes the order: at most one copy or two fragment reads behind any
MFMA, nothing else.

Loop structure (operand A: m-contiguous tile read with transposed LDS reads, operand B:
k-contiguous tile read with ds_read_b128; ring of 4 LDS stages of 32 KB, stage = A tile then B
tile; the body is unrolled over the 4 stages so that every LDS offset is an immediate):

  step k, stage s = k % 4
    MFMA  0..15  use fragments f0 = (stage s, contraction 0..15), read during step k-1
    MFMA 16..31  use fragments f1 = (stage s, contraction 16..31), read behind MFMA 0..7
    copies of step k+3 -> stage (s+3) % 4 (read during step k-1, free since the barrier of
      that step): A tile behind MFMA 1, 5, 8, 10, B tile behind MFMA 19, 22, 25, 28
    behind MFMA 12: wait until this wavefront's copies of step k+1 have landed
      (vmcnt(12): step k+2 and the A half of step k+3 may stay in flight) and its reads of
      stage s have returned, barrier; then f0 of step k+1 is read behind MFMA 12..17, each
      read into registers whose last MFMA has been issued.
  Copies are issued for every step, including the last three whose data nobody reads: their
  source is clamped to the last valid step, which keeps the loop free of branches and the
  vmcnt arithmetic uniform.

CT_GEMM_FRESH_LOOP starts from C = 0 (the first step's first MFMAs take the constant, no accumulator is
cleared) and its copies of steps 0..2 may be older than an epilogue's stores: vmcnt counts in order, so a
first iteration of its own waits for no more than the copies it needs. With at least 51 stores behind
those copies (CT_GEMM_FRESH_LOOP_BEHIND_STORES), vmcnt(63), the largest there is, holds whatever is older
than the youngest 63: step 1's (8 copies of step 2, the stores, 4 copies of step 3 follow them) and, a step
later, step 2's; only step 2 waits for the stores, for it needs the copies of step 3 behind them.

An operand whose rows start at any multiple of 2 bytes (a head of odd vocabulary) cannot be copied that way: the copies
move aligned 16 bytes. CT_GEMM_VIA_A_LOOP and CT_GEMM_VIA_B_LOOP take it through registers instead, in the slots of operand
A's copies (the other operand's copies keep the late ones): a chunk of step k + 1, on its way for two steps, goes to
LDS, and the load of step k + 3 into the registers that this frees follows it. Two sets of 16 registers, as many
loads and copies in flight as before; the first steps' loads are issued in the statement itself, behind
the other operand's copies, so the first iteration counts less in flight. The rows of B, of which a step takes 64 bytes, are
read 128 bytes at a time: an odd step k stores the chunks of steps k + 1 and k + 2 and loads those of k + 3 and k + 4
(64 bytes at a time the gradients of 102 rows x 173037, d = 2944 took 819 us for 677, of 1081 x 58435, d = 4608 1970 for 1678;
from an aligned copy, made in 342 and 186 us, they take 587 and 1466).

Fixed registers (declared as clobbers): v[144:175] what such loads fill, v[176:239] fragments, v[240:249] fragment addresses
+ 64 KB (v250 the thread's place in the upper stages), s[40:41] / s[42:43] copy sources of A / B, s44 step counter,
s45-s46 temporaries.

Run ``python gen_gemm_asm.py > ct_gemm_asm.inc`` after editing; the output is committed.
"""

STAGE = 32768
VIA, F0A, F0B, F1A, F1B, HI = 144, 176, 192, 208, 224, 240
SRC = ("s[40:41]", "s[42:43]")
ACC = lambda i, j: "%%%d" % (4 * i + j)
PTR_A, PTR_B, STRIDE_A, STEPS, LDS_WAVE = "%16", "%17", "%18", "%19", "%20"
ADDR_A = lambda second, i: 21 + 4 * second + i
ADDR_B = lambda ks: 29 + ks
VOFF = lambda operand, n: "%%%d" % (31 + 4 * operand + n)
THREAD = ("%39", "%43")           # LDS address of the thread's first chunk of stage 0, by the operand through registers


def addr(operand_index, stage, offset):
    """register and immediate of an LDS read at (address operand) + stage * STAGE + offset"""
    if stage < 2:
        return "%%%d" % operand_index, stage * STAGE + offset
    return "v%d" % (HI + operand_index - 21), (stage - 2) * STAGE + offset


def frag_reads(stage, ks):
    """the 12 reads of the fragments (stage, ks), keyed by the fragment they fill"""
    fa, fb = (F0A, F0B) if ks == 0 else (F1A, F1B)
    out = {}
    for i in range(4):
        reads = []
        for second in range(2):
            reg, imm = addr(ADDR_A(second, i), stage, ks * 8192)
            lo = fa + 4 * i + 2 * second
            reads.append("ds_read_b64_tr_b16 v[%d:%d], %s offset:%d" % (lo, lo + 1, reg, imm))
        out["a%d" % i] = reads
    for j in range(4):
        reg, imm = addr(ADDR_B(ks), stage, j * 2048)
        lo = fb + 4 * j
        out["b%d" % j] = ["ds_read_b128 v[%d:%d], %s offset:%d" % (lo, lo + 3, reg, imm)]
    return out


def mfma(m, from_zero=False):
    ks, r = divmod(m, 16)
    i, j = divmod(r, 4)
    fa, fb = (F0A, F0B) if ks == 0 else (F1A, F1B)
    return "v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], v[%d:%d], %s" % (
        ACC(i, j), fa + 4 * i, fa + 4 * i + 3, fb + 4 * j, fb + 4 * j + 3, "0" if from_zero and ks == 0 else ACC(i, j))


def copy(operand, n, stage):
    dst = stage * STAGE + operand * 16384 + n * 4096
    return ["s_add_u32 m0, %s, %d" % (LDS_WAVE, dst), "s_nop 0",
            "global_load_lds_dwordx4 %s, %s" % (VOFF(operand, n), SRC[operand])]


def load(operand, n, registers):
    return "global_load_dwordx4 v[%d:%d], %s, %s" % (registers + 4 * n, registers + 4 * n + 3, VOFF(operand, n), SRC[operand])


def to_lds(operand, n, registers, stage):
    where, low = (THREAD[operand], stage) if stage < 2 else ("v%d" % (HI + 10), stage - 2)
    return "ds_write_b128 %s, v[%d:%d] offset:%d" % (where, registers + 4 * n, registers + 4 * n + 3,
                                                     low * STAGE + operand * 16384 + n * (4096, 2048)[operand])


ADVANCE_A = ["s_cmp_lt_u32 s44, " + STEPS, "s_cselect_b32 s45, %s, 0" % STRIDE_A, "s_add_u32 s40, s40, s45", "s_addc_u32 s41, s41, 0"]
ADVANCE = [
    "s_cmp_lt_u32 s44, " + STEPS,
    "s_cselect_b32 s45, %s, 0" % STRIDE_A,
    "s_cselect_b32 s46, 64, 0",
    "s_add_u32 s40, s40, s45",
    "s_addc_u32 s41, s41, 0",
    "s_add_u32 s42, s42, s46",
    "s_addc_u32 s43, s43, 0",
    "s_add_u32 s44, s44, 1",
]


def advance_pair(next_step):
    """the source of B's pairs of steps, one pair on if that begins ahead of the end at step `next_step` (a register)"""
    return ["s_cmp_lt_u32 %s, %s" % (next_step, STEPS), "s_cselect_b32 s46, 128, 0", "s_add_u32 s42, s42, s46", "s_addc_u32 s43, s43, 0"]


def step(u, from_zero=False, in_flight=12, via=None, behind_chunk=15):
    """step u % 4 of an iteration; in_flight: how many copies (and stores) may be when step u + 1's have landed;
    via: the operand that comes through registers, behind_chunk: how many loads and copies follow a chunk's load"""
    stage, nxt, dst = u, (u + 1) & 3, (u + 3) & 3
    f1 = frag_reads(stage, 1)
    f0n = frag_reads(nxt, 0)
    behind = {m: [] for m in range(32)}
    # f1 of this stage: all of its registers are free (their MFMAs belong to the last step)
    for m, keys in {0: ["a0"], 2: ["b0", "b1"], 3: ["b2", "b3"], 4: ["a1"], 6: ["a2"], 7: ["a3"]}.items():
        for key in keys:
            behind[m] += f1[key]
    if via is None:
        for m, n in {1: 0, 5: 1, 8: 2, 10: 3}.items():
            behind[m] += copy(0, n, dst)
    elif via == 0:
        through = VIA + 16 * (nxt & 1)
        for m, n in {1: 0, 5: 1, 8: 2, 10: 3}.items():
            behind[m] += ["s_waitcnt vmcnt(%d)" % behind_chunk, to_lds(0, n, through, nxt), load(0, n, through)]
    elif u & 1:
        for n, m in enumerate((1, 3, 5, 7, 8, 9, 10, 11)):
            behind[m] += ["s_waitcnt vmcnt(%d)" % behind_chunk, to_lds(1, n, VIA, nxt), load(1, n, VIA)]
    behind[12] += ["s_waitcnt vmcnt(%d)" % in_flight, "s_waitcnt lgkmcnt(0)", "s_barrier"]
    # f0 of the next step: a0..a2 are free after MFMA 11, b_j after MFMA 12 + j, a3 after MFMA 15
    for m, keys in {12: ["a0"], 13: ["a1"], 14: ["a2"], 15: ["b0", "b1"], 16: ["b2", "b3"], 17: ["a3"]}.items():
        for key in keys:
            behind[m] += f0n[key]
    for m, n in {19: 0, 22: 1, 25: 2, 28: 3}.items():
        behind[m] += copy(0 if via == 1 else 1, n, dst)
    if via == 1:
        behind[29] += ADVANCE_A + ["s_add_u32 s44, s44, 1"] + (advance_pair("s44") if u & 1 else [])
    else:
        behind[29] += ADVANCE
    lines = ["s_waitcnt lgkmcnt(0)"]
    for m in range(32):
        lines.append(mfma(m, from_zero))
        lines += behind[m]
    return lines


def gemm_loop(fresh=False, behind_stores=False, via=None):
    lines = ["s_mov_b64 s[40:41], " + PTR_A, "s_mov_b64 s[42:43], " + PTR_B, "s_mov_b32 s44, 4"]
    # (the source of an operand through registers is that of step 0)
    if via == 0:
        for registers in (F1A, VIA + 16, VIA):
            lines += [load(0, n, registers) for n in range(4)] + ["s_add_u32 s40, s40, " + STRIDE_A, "s_addc_u32 s41, s41, 0"]
    elif via == 1:
        lines += [load(1, n, F1A) for n in range(8)] + ["s_add_u32 s42, s42, 128", "s_addc_u32 s43, s43, 0"]
        lines += [load(1, n, VIA) for n in range(8)] + advance_pair("s44")
    if via is not None:
        lines.append("v_add_u32 v%d, 0x10000, %s" % (HI + 10, THREAD[via]))
    for k in range(10):
        lines.append("v_add_u32 v%d, 0x10000, %%%d" % (HI + k, 21 + k))
    if via is not None:
        # step 0 (the first pair) and all copies have landed
        lines += ["s_waitcnt vmcnt(8)"] + [to_lds(via, n, F1A, 0) for n in range(4 + 4 * via)] + ["s_waitcnt lgkmcnt(0)", "s_barrier"]
    first = frag_reads(0, 0)
    for key in ["a0", "b0", "b1", "b2", "b3", "a1", "a2", "a3"]:
        lines += first[key]
    first_iteration = fresh or via is not None
    if first_iteration:
        for u in range(4):
            lines += step(u, from_zero=fresh and u == 0, in_flight=63 if behind_stores and u < 2 else 12, via=via,
                          behind_chunk=(7, 11, 15, 15)[u])
        lines += ["s_sub_u32 s45, s44, 4", "s_cmp_lt_u32 s45, " + STEPS, "s_cbranch_scc0 ct_gemm_done_%="]
    lines.append("ct_gemm_loop_%=:")
    for u in range(4):
        lines += step(u, via=via)
    lines += ["s_sub_u32 s45, s44, 4", "s_cmp_lt_u32 s45, " + STEPS, "s_cbranch_scc1 ct_gemm_loop_%="]
    if first_iteration:
        lines.append("ct_gemm_done_%=:")
    # drain: nothing in flight, every wavefront done with the LDS tiles, MFMA results readable
    lines += ["s_waitcnt vmcnt(0)", "s_waitcnt lgkmcnt(0)", "s_barrier", "s_nop 15", "s_nop 7"]
    return lines


# ---------------------------------------------------------------------------
# The 128 x 128 tile (2 x 2 blocks per wavefront; ring of 4 LDS stages of 16 KB)
# ---------------------------------------------------------------------------
# 8 MFMAs a step are too few to read a step's second half of fragments behind its first, so all fragments
# of step k + 1 are read, into the other of two register sets, behind the MFMAs of step k:
#
#   step k, stage s = k % 4
#     the fragments of step k have arrived (they were read during step k-1: stage s is free now)
#     MFMA 0; behind it: this wavefront's copies of step k+1 have landed (vmcnt(8): steps k+2 and
#       k+3 may stay in flight), barrier
#     reads of step k+1's fragments behind MFMA 1..6, copies of step k+4 -> stage s behind MFMA 1, 3, 5, 7
#
# An operand through registers (`via`): a chunk of step k+2, loaded in step k-2, goes to LDS behind MFMA 1 or 3, the load
# of step k+4 into its registers follows. It is there in front of the next step's barrier, behind which step k+2's
# fragments are read. B's rows are read 128 bytes at a time here too: an even step k stores the chunks of steps k+2 and
# k+3 and loads those of k+4 and k+5. Two sets of 8 registers.
#
# Fixed registers (clobbers): v[64:95], v[96:127] the two sets, s[40:41] / s[42:43], s44, s45-s46 as above. With an
# operand through registers v[48:79], v[80:111], v[112:127] the loads': the compiler gives a kernel of two workgroups
# 128 vector registers and 128 accumulation registers, and one more of the first would be one workgroup less.
SMALL_STAGE = 16384
SMALL_SETS = {None: (64, 96), 0: (48, 80), 1: (48, 80)}
SMALL_VIA = 112
SMALL_ACC = lambda i, j: "%%%d" % (2 * i + j)
SMALL_IN = {name: "%%%d" % (4 + k) for k, name in enumerate(
    ["src_a", "src_b", "stride_a", "steps", "lds_wave", "a00", "a01", "a10", "a11", "b0", "b1", "va0", "va1", "vb0", "vb1",
     "vb2", "vb3"])}
SMALL_THREAD = ("%19", "%21")


def small_frag(first, operand, ks, i):
    return first + 16 * ks + 8 * operand + 4 * i


def small_reads(stage, first):
    """the 12 reads of a step's fragments, in the order of their use"""
    out = []
    for ks in range(2):
        for i in range(2):
            for second in range(2):
                lo = small_frag(first, 0, ks, i) + 2 * second
                out.append("ds_read_b64_tr_b16 v[%d:%d], %s offset:%d" % (
                    lo, lo + 1, SMALL_IN["a%d%d" % (second, i)], stage * SMALL_STAGE + ks * 4096))
            lo = small_frag(first, 1, ks, i)
            out.append("ds_read_b128 v[%d:%d], %s offset:%d" % (
                lo, lo + 3, SMALL_IN["b%d" % ks], stage * SMALL_STAGE + i * 2048))
    return out


def small_copy(operand, n, stage):
    return ["s_add_u32 m0, %s, %d" % (SMALL_IN["lds_wave"], stage * SMALL_STAGE + operand * 8192 + n * 4096), "s_nop 0",
            "global_load_lds_dwordx4 %s, %s" % (SMALL_IN["v%s%d" % ("ab"[operand], n)], SRC[operand])]


def small_load(operand, n, registers):
    return "global_load_dwordx4 v[%d:%d], %s, %s" % (registers + 4 * n, registers + 4 * n + 3,
                                                     SMALL_IN["v%s%d" % ("ab"[operand], n)], SRC[operand])


def small_to_lds(operand, n, registers, stage):
    return "ds_write_b128 %s, v[%d:%d] offset:%d" % (SMALL_THREAD[operand], registers + 4 * n, registers + 4 * n + 3,
                                                     stage * SMALL_STAGE + operand * 8192 + n * (4096, 2048)[operand])


def small_names(line):
    return line.replace(STRIDE_A, SMALL_IN["stride_a"]).replace(STEPS, SMALL_IN["steps"])


def small_step(u, via=None, behind_chunk=7):
    stage, current, other = u, SMALL_SETS[via][u & 1], SMALL_SETS[via][(u + 1) & 1]
    reads = small_reads((u + 1) & 3, other)
    behind = {m: [] for m in range(8)}
    if via == 1:
        behind[0] = ADVANCE_A + ([] if u & 1 else advance_pair("s44")) + ["s_add_u32 s44, s44, 1"]
    else:
        behind[0] = list(ADVANCE)
    behind[0] = [small_names(ln) for ln in behind[0]] + ["s_waitcnt vmcnt(8)", "s_barrier"]
    for m in range(1, 7):
        behind[m] += reads[2 * m - 2:2 * m]
    if via == 0:
        through = SMALL_VIA + 8 * (u & 1)
        for m, n in {1: 0, 3: 1}.items():
            behind[m] += ["s_waitcnt vmcnt(%d)" % behind_chunk, small_to_lds(0, n, through, (u + 2) & 3), small_load(0, n, through)]
    elif via == 1 and not u & 1:
        for n in range(4):
            behind[1 + n] += ["s_waitcnt vmcnt(%d)" % behind_chunk, small_to_lds(1, n, SMALL_VIA, (u + 2) & 3),
                              small_load(1, n, SMALL_VIA)]
    early, late = (1, 0) if via == 1 else (0, 1)
    for m, (operand, n) in {1: (early, 0), 3: (early, 1), 5: (late, 0), 7: (late, 1)}.items():
        if operand != via:
            behind[m] += small_copy(operand, n, stage)
    lines = ["s_waitcnt lgkmcnt(0)"]
    for m in range(8):
        ks, i, j = m >> 2, (m >> 1) & 1, m & 1
        a, b = small_frag(current, 0, ks, i), small_frag(current, 1, ks, j)
        lines.append("v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], v[%d:%d], %s" % (
            SMALL_ACC(i, j), a, a + 3, b, b + 3, SMALL_ACC(i, j)))
        lines += behind[m]
    return lines


def small_loop(via=None):
    lines = ["s_mov_b64 s[40:41], " + SMALL_IN["src_a"], "s_mov_b64 s[42:43], " + SMALL_IN["src_b"], "s_mov_b32 s44, 4"]
    if via is not None:     # (the source of an operand through registers is that of step 0)
        first = SMALL_SETS[via][1]
        if via == 0:
            for k, registers in enumerate((first, first + 8, SMALL_VIA, SMALL_VIA + 8)):
                lines += ["s_add_u32 s40, s40, " + SMALL_IN["stride_a"], "s_addc_u32 s41, s41, 0"] if k else []
                lines += [small_load(0, n, registers) for n in range(2)]
        else:
            lines += [small_load(1, n, first) for n in range(4)] + ["s_add_u32 s42, s42, 128", "s_addc_u32 s43, s43, 0"]
            lines += [small_load(1, n, SMALL_VIA) for n in range(4)]
        # steps 0 and 1 and all copies have landed
        lines.append("s_waitcnt vmcnt(4)")
        lines += [small_to_lds(1, n, first, 0) for n in range(4)] if via else [
            small_to_lds(0, n, first + 8 * k, k) for k in range(2) for n in range(2)]
        lines += ["s_waitcnt lgkmcnt(0)", "s_barrier"]
    lines += small_reads(0, SMALL_SETS[via][0])
    # (s44 has advanced by 4: the steps done are s44 - 4; the last one read fragments that nobody uses)
    more = ["s_sub_u32 s45, s44, 4", "s_cmp_lt_u32 s45, " + SMALL_IN["steps"]]
    if via is not None:
        for u in range(4):
            lines += small_step(u, via, (3, 7 if via else 5, 7, 7)[u])
        lines += more + ["s_cbranch_scc0 ct_gemm_small_done_%="]
    lines.append("ct_gemm_small_loop_%=:")
    for u in range(4):
        lines += small_step(u, via)
    lines += more + ["s_cbranch_scc1 ct_gemm_small_loop_%="]
    if via is not None:
        lines.append("ct_gemm_small_done_%=:")
    lines += ["s_waitcnt vmcnt(0)", "s_waitcnt lgkmcnt(0)", "s_barrier", "s_nop 15", "s_nop 7"]
    return lines


def emit(lines, name):
    body = " \\\n".join('  "%s\\n\\t"' % ln for ln in lines)
    return "#define %s \\\n%s\n" % (name, body)


def clobbers(first, end):
    regs = ["v%d" % r for r in range(first, end)] + ["s%d" % r for r in range(40, 47)]
    return ", ".join('"%s"' % r for r in regs)


if __name__ == "__main__":
    print("// Generated by gen_gemm_asm.py -- do not edit by hand.")
    print(emit(gemm_loop(), "CT_GEMM_LOOP"))
    print(emit(gemm_loop(fresh=True), "CT_GEMM_FRESH_LOOP"))
    print(emit(gemm_loop(fresh=True, behind_stores=True), "CT_GEMM_FRESH_LOOP_BEHIND_STORES"))
    print("#define CT_GEMM_LOOP_CLOBBERS %s" % clobbers(F0A, HI + 10))
    print(emit(gemm_loop(fresh=True, via=0), "CT_GEMM_VIA_A_LOOP"))
    print(emit(gemm_loop(via=1), "CT_GEMM_VIA_B_LOOP"))
    print("#define CT_GEMM_VIA_LOOP_CLOBBERS %s" % clobbers(VIA, HI + 11))
    print(emit(small_loop(), "CT_GEMM_SMALL_LOOP"))
    print("#define CT_GEMM_SMALL_LOOP_CLOBBERS %s" % clobbers(SMALL_SETS[None][0], SMALL_SETS[None][1] + 32))
    print(emit(small_loop(via=0), "CT_GEMM_SMALL_VIA_A_LOOP"))
    print(emit(small_loop(via=1), "CT_GEMM_SMALL_VIA_B_LOOP"))
    print("#define CT_GEMM_SMALL_VIA_LOOP_CLOBBERS %s" % clobbers(SMALL_SETS[0][0], SMALL_VIA + 16))
