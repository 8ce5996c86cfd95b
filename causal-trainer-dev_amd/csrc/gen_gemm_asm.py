"""Generates ct_gemm_asm.inc: the hand-scheduled main loops of the 256 x 256 and 128 x 128 GEMM tiles.

One wavefront runs on each SIMD, so whatever the wavefront issues between two MFMAs must fit
into the 32 cycles the matrix pipe is busy with the first of them, or the pipe drains. A
global -> LDS copy costs about 23 cycles to issue and an LDS fragment read 4 to 8; issued in
bursts (as the compiler schedules them) they stall the MFMA stream for hundreds of cycles per
k-step. The sequence below fixes the order: at most one copy or two fragment reads behind any
MFMA, nothing else.

Loop structure (operand A: m-contiguous tile read with transposed LDS reads, operand B:
k-contiguous tile read with ds_read_b128). LDS holds four stages of A, one per step, and behind them two stages of
B, one per pair of steps: a step takes 64 bytes of each row of B, half of a cache line, and the memory system
serves a copy of whole lines 1.2 to 1.8 times as fast (a copy loop of 8 KB of A and 8 KB of B a step from 400 workgroups, 61.5
us in pieces of 64 bytes, 49.9 of 128). The body is unrolled over four steps so that every LDS offset is an immediate.

  step k, A stage s = k % 4, B stage k / 2 % 2
    MFMA  0..15  use fragments f0 = (step k, contraction 0..15), read during step k-1
    MFMA 16..31  use fragments f1 = (step k, contraction 16..31), read behind MFMA 0..7
    copies of A's step k+3 -> stage (s+3) % 4 (read during step k-1, free since the barrier of
      that step) behind MFMA 1, 5, 8, 10
    behind MFMA 12: wait until this wavefront's copies of step k+1 have landed and its reads of step k have returned,
      barrier; then f0 of step k+1 is read behind MFMA 12..17, each read into registers whose last MFMA has been
      issued. May stay in flight: in an even step A's steps k+2 and k+3 and the pair behind (vmcnt(16); step k+1 is
      of the same pair), in an odd one A's (vmcnt(8)).
    odd steps: copies of the pair of steps k+3 and k+4 into the stage that this step's barrier has freed, behind
      MFMA 18 to 28
  Copies are issued for every step, including the last three whose data nobody reads: their
  source is clamped to the last valid step or pair, which keeps the loop free of branches and the
  vmcnt arithmetic uniform.

CT_GEMM_FRESH_LOOP starts from C = 0 (the first step's first MFMAs take the constant, no accumulator is
cleared) and its copies of steps 0..2 and pairs 0 and 1 may be older than an epilogue's stores: vmcnt counts in order, so
a first iteration of its own waits for no more than the copies it needs. With at least 55 stores behind
those copies (CT_GEMM_FRESH_LOOP_BEHIND_STORES), vmcnt(63), the largest there is, holds whatever is older
than the youngest 63: A's step 1 (step 2, pair 1, the stores and step 3 follow it) and, a step later, pair 1 (the
stores, steps 3 and 4); only step 2 waits for the stores, for it needs the copies of step 3 behind them.

An operand whose rows start at any multiple of 2 bytes (a head of odd vocabulary) cannot be copied that way: the copies
move aligned 16 bytes. CT_GEMM_VIA_A_LOOP and CT_GEMM_VIA_B_LOOP take it through registers instead, in the slots of operand
A's copies (the other operand's copies keep the late ones): a chunk of step k + 1, on its way for two steps, goes to
LDS, and the load of step k + 3 into the registers that this frees follows it; of B an odd step stores the chunks of the
pair k + 1, k + 2 and loads those of k + 3, k + 4. 32 registers, as many loads and copies in flight as
before; the first steps' loads are issued in the statement itself, behind the other operand's copies, so the first
iteration counts less in flight. (In pieces of 64 bytes the gradients of 102 rows x 173037, d = 2944 took 819 us for 677, of
1081 x 58435, d = 4608 1970 for 1678.)

Fixed registers (declared as clobbers): v[144:175] what such loads fill, v[176:239] fragments, s[40:41] / s[42:43] copy
sources of A / B, s44 step counter, s45-s46 temporaries.

Run ``python gen_gemm_asm.py > ct_gemm_asm.inc`` after editing; the output is committed.
"""

A_STAGE, B_AT, B_STAGE = 16384, 65536, 32768
VIA, F0A, F0B, F1A, F1B = 144, 176, 192, 208, 224
SRC = ("s[40:41]", "s[42:43]")
ACC = lambda i, j: "%%%d" % (4 * i + j)
PTR_A, PTR_B, STRIDE_A, STEPS, LDS_WAVE = "%16", "%17", "%18", "%19", "%20"
ADDR_A = lambda second, i: "%%%d" % (21 + 4 * second + i)
ADDR_B = lambda ks: "%%%d" % (29 + ks)          # ks: of the four of a pair
VOFF = (lambda n: "%%%d" % (33 + n), lambda n: "%%%d" % (37 + n))
THREAD = "%45"      # the thread's first 16 bytes of the first stage of the operand through registers


def frag_reads(stage, ks):
    """the 12 reads of the fragments (step `stage` of four, ks), keyed by the fragment they fill"""
    fa, fb = (F0A, F0B) if ks == 0 else (F1A, F1B)
    out = {}
    for i in range(4):
        reads = []
        for second in range(2):
            lo = fa + 4 * i + 2 * second
            reads.append("ds_read_b64_tr_b16 v[%d:%d], %s offset:%d" % (lo, lo + 1, ADDR_A(second, i), stage * A_STAGE + ks * 8192))
        out["a%d" % i] = reads
    for j in range(4):
        lo = fb + 4 * j
        out["b%d" % j] = ["ds_read_b128 v[%d:%d], %s offset:%d" % (
            lo, lo + 3, ADDR_B(2 * (stage & 1) + ks), (stage >> 1) * B_STAGE + j * 4096)]
    return out


def mfma(m, from_zero=False):
    ks, r = divmod(m, 16)
    i, j = divmod(r, 4)
    fa, fb = (F0A, F0B) if ks == 0 else (F1A, F1B)
    return "v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], v[%d:%d], %s" % (
        ACC(i, j), fa + 4 * i, fa + 4 * i + 3, fb + 4 * j, fb + 4 * j + 3, "0" if from_zero and ks == 0 else ACC(i, j))


def copy(operand, n, stage):
    """chunk n of a stage of A, or of a pair's stage of B"""
    dst = (B_AT + stage * B_STAGE if operand else stage * A_STAGE) + n * 4096
    return ["s_add_u32 m0, %s, %d" % (LDS_WAVE, dst), "s_nop 0",
            "global_load_lds_dwordx4 %s, %s" % (VOFF[operand](n), SRC[operand])]


def load(operand, n, registers):
    return "global_load_dwordx4 v[%d:%d], %s, %s" % (registers + 4 * n, registers + 4 * n + 3, VOFF[operand](n), SRC[operand])


def to_lds(operand, n, registers, stage):
    return "ds_write_b128 %s, v[%d:%d] offset:%d" % (THREAD, registers + 4 * n, registers + 4 * n + 3,
                                                     stage * (B_STAGE if operand else A_STAGE) + n * 4096)


# Where the sources go next: A's is that of step s44, unless that is past the end; B's that of the pair that begins with it.
ADVANCE_A = ["s_cmp_lt_u32 s44, " + STEPS, "s_cselect_b32 s45, %s, 0" % STRIDE_A, "s_add_u32 s40, s40, s45", "s_addc_u32 s41, s41, 0"]
ADVANCE_B = ["s_cmp_lt_u32 s44, " + STEPS, "s_cselect_b32 s46, 128, 0", "s_add_u32 s42, s42, s46", "s_addc_u32 s43, s43, 0"]
NEXT_STEP = ["s_add_u32 s44, s44, 1"]


def step(u, from_zero=False, behind_stores=False, via=None, behind_chunk=15):
    """step u % 4 of an iteration; behind_stores: the epilogue's may lie behind the copies that it waits for; via: the
    operand that comes through registers, behind_chunk: how many loads and copies follow a chunk's load"""
    stage, nxt, dst, odd = u, (u + 1) & 3, (u + 3) & 3, u & 1
    f1 = frag_reads(stage, 1)
    f0n = frag_reads(nxt, 0)
    behind = {m: [] for m in range(32)}
    # f1 of this stage: all of its registers are free (their MFMAs belong to the last step)
    for m, keys in {0: ["a0"], 2: ["b0", "b1"], 3: ["b2", "b3"], 4: ["a1"], 6: ["a2"], 7: ["a3"]}.items():
        for key in keys:
            behind[m] += f1[key]
    chunk_wait = "s_waitcnt vmcnt(%d)" % behind_chunk
    if via == 1:
        for n, m in enumerate((1, 3, 5, 7, 8, 9, 10, 11) if odd else ()):
            behind[m] += [chunk_wait, to_lds(1, n, VIA, nxt >> 1), load(1, n, VIA)]
        for n, m in enumerate((19, 22, 25, 28)):
            behind[m] += copy(0, n, dst)
        landed = 12
    else:
        through = VIA + 16 * (nxt & 1)
        for n, m in enumerate((1, 5, 8, 10)):
            behind[m] += copy(0, n, dst) if via is None else [chunk_wait, to_lds(0, n, through, nxt), load(0, n, through)]
        for n, m in enumerate((18, 19, 21, 22, 24, 25, 27, 28) if odd else ()):
            behind[m] += copy(1, n, stage >> 1)
        landed = 63 if behind_stores else 8 if odd else 16 if via is None else None
    if landed is not None:
        behind[12].append("s_waitcnt vmcnt(%d)" % landed)
    behind[12] += ["s_waitcnt lgkmcnt(0)", "s_barrier"]
    # f0 of the next step: a0..a2 are free after MFMA 11, b_j after MFMA 12 + j, a3 after MFMA 15
    for m, keys in {12: ["a0"], 13: ["a1"], 14: ["a2"], 15: ["b0", "b1"], 16: ["b2", "b3"], 17: ["a3"]}.items():
        for key in keys:
            behind[m] += f0n[key]
    behind[29] += ADVANCE_A + NEXT_STEP
    behind[30] += ADVANCE_B if odd else []
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
        lines += [load(1, n, VIA) for n in range(8)] + ADVANCE_B
    if via is not None:
        # step 0 (the first pair) and all copies have landed
        lines += ["s_waitcnt vmcnt(8)"] + [to_lds(via, n, F1A, 0) for n in range(4 + 4 * via)] + ["s_waitcnt lgkmcnt(0)", "s_barrier"]
    first = frag_reads(0, 0)
    for key in ["a0", "b0", "b1", "b2", "b3", "a1", "a2", "a3"]:
        lines += first[key]
    first_iteration = fresh or via is not None
    if first_iteration:
        for u in range(4):
            lines += step(u, from_zero=fresh and u == 0, behind_stores=behind_stores and u < 2, via=via,
                          behind_chunk=((7, 7, 15, 15), (0, 11, 0, 15))[via or 0][u])
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
# The 128 x 128 tile (2 x 2 blocks per wavefront; four stages of A of 8 KB, two of B of 16 KB; or eight and four)
# ---------------------------------------------------------------------------
# 8 MFMAs a step are too few to read a step's second half of fragments behind its first, so all fragments
# of step k + 1 are read, into the other of two register sets, behind the MFMAs of step k:
#
#   step k, A stage s = k % 4, B stage k / 2 % 2
#     the fragments of step k have arrived (they were read during step k-1: stage s is free now, in an odd step B's too)
#     MFMA 0; behind it: this wavefront's copies of step k+1 have landed, barrier. May stay in flight: in an even step the
#       pair behind (4 copies) and A's steps k+2 and k+3 (2 each; vmcnt(8)), in an odd one A's only (vmcnt(4))
#     reads of step k+1's fragments behind MFMA 1..6, in an odd step copies of the pair of steps k+3 and k+4 behind MFMA 1 to
#       4, then those of A's step k+4 -> stage s behind MFMA 5, 7
#
# With eight stages of A and four of B (RING = 8, for a workgroup that has its compute unit to itself) the copies of A's
# step k+8 and in odd steps of the pair of steps k+7 and k+8 take their places: six steps on their way instead of
# two. A body of eight steps, with an end in the middle.
#
# An operand through registers (`via`): a chunk of step k+2, loaded in step k-2, goes to LDS behind MFMA 1 or 3, the load
# of step k+4 into its registers follows. It is there in front of the next step's barrier, behind which step k+2's
# fragments are read (an odd step's barrier has let it land already). Of B an even step k stores the chunks of the pair
# k+2, k+3 and loads those of k+4, k+5. 16 registers; with eight stages 32, the load is that of step k+6.
#
# Fixed registers (clobbers): v[64:95], v[96:127] the two sets, s[40:41] / s[42:43], s44, s45-s46 as above. With an
# operand through registers v[48:79], v[80:111], v[112:127] the loads': the compiler gives a kernel of two workgroups
# 128 vector registers and 128 accumulation registers, and one more of the first would be one workgroup less.
SMALL_A_STAGE, SMALL_B_STAGE = 8192, 16384
SMALL_SETS = {None: (64, 96), 0: (48, 80), 1: (48, 80)}
SMALL_VIA = 112
SMALL_ACC = lambda i, j: "%%%d" % (2 * i + j)
SMALL_IN = {name: "%%%d" % (4 + k) for k, name in enumerate(
    ["src_a", "src_b", "stride_a", "steps", "lds_wave", "a00", "a01", "a10", "a11", "b0", "b1", "b2", "b3", "va0", "va1",
     "vb0", "vb1", "vb2", "vb3", "thread"])}


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
                    lo, lo + 1, SMALL_IN["a%d%d" % (second, i)], stage * SMALL_A_STAGE + ks * 4096))
            lo = small_frag(first, 1, ks, i)
            out.append("ds_read_b128 v[%d:%d], %s offset:%d" % (
                lo, lo + 3, SMALL_IN["b%d" % (2 * (stage & 1) + ks)], (stage >> 1) * SMALL_B_STAGE + i * 4096))
    return out


def small_voff(operand, n):
    return SMALL_IN["v%s%d" % ("ab"[operand], n)]


def small_copy(operand, n, stage, ring):
    dst = (ring * SMALL_A_STAGE + stage * SMALL_B_STAGE if operand else stage * SMALL_A_STAGE) + n * 4096
    return ["s_add_u32 m0, %s, %d" % (SMALL_IN["lds_wave"], dst), "s_nop 0",
            "global_load_lds_dwordx4 %s, %s" % (small_voff(operand, n), SRC[operand])]


def small_load(operand, n, registers):
    return "global_load_dwordx4 v[%d:%d], %s, %s" % (registers + 4 * n, registers + 4 * n + 3, small_voff(operand, n), SRC[operand])


def small_to_lds(operand, n, registers, stage):
    return "ds_write_b128 %s, v[%d:%d] offset:%d" % (SMALL_IN["thread"], registers + 4 * n, registers + 4 * n + 3,
                                                     stage * (SMALL_B_STAGE if operand else SMALL_A_STAGE) + n * 4096)


def small_names(lines):
    return [line.replace(STRIDE_A, SMALL_IN["stride_a"]).replace(STEPS, SMALL_IN["steps"]) for line in lines]


def small_step(u, via=None, ring=4, behind_chunk=None):
    odd, current, other = u & 1, SMALL_SETS[via][u & 1], SMALL_SETS[via][(u + 1) & 1]
    reads = small_reads((u + 1) % ring, other)
    behind = {m: [] for m in range(8)}
    # Sources: A's of step k + ring (k + 6 through registers with eight stages); B's of the pair that begins with step
    # k + 4 through registers, else, behind its copies, with step k + ring + 1.
    if via == 0 and ring == 8:
        behind[0] = ["s_sub_u32 s45, s44, 2", "s_cmp_lt_u32 s45, " + STEPS] + ADVANCE_A[1:]
    else:
        behind[0] = list(ADVANCE_A)
    behind[0] = small_names(behind[0] + (ADVANCE_B if via == 1 and not odd else []) + NEXT_STEP)
    landed = {(None, 4): (8, 4), (None, 8): (24, 20), (0, 4): (None, 2), (0, 8): (None, None), (1, 4): (8, 8)}[via, ring][odd]
    if landed is not None:
        behind[0].append("s_waitcnt vmcnt(%d)" % landed)
    behind[0].append("s_barrier")
    for m in range(1, 7):
        behind[m] += reads[2 * m - 2:2 * m]
    if behind_chunk is None:
        behind_chunk = 15 if ring == 8 else 7
    chunk_wait = ["s_waitcnt vmcnt(%d)" % behind_chunk]
    if via == 1:
        for n in range(0 if odd else 4):
            behind[1 + n] += chunk_wait + [small_to_lds(1, n, SMALL_VIA, ((u + 2) & 3) >> 1), small_load(1, n, SMALL_VIA)]
        for n, m in enumerate((5, 7)):
            behind[m] += small_copy(0, n, u, ring)
    else:
        through = SMALL_VIA + 8 * ((u + 2) % (ring // 2))
        for n, m in enumerate((5, 7) if via is None else (1, 3)):
            behind[m] += small_copy(0, n, u, ring) if via is None else ([] if odd and ring == 4 else chunk_wait) + [
                small_to_lds(0, n, through, (u + 2) % ring), small_load(0, n, through)]
        for n in range(4 if odd else 0):
            behind[(1 if via is None else 4) + n] += small_copy(1, n, u >> 1, ring)
        behind[7] += small_names(ADVANCE_B) if odd else []
    lines = ["s_waitcnt lgkmcnt(0)"]
    for m in range(8):
        ks, i, j = m >> 2, (m >> 1) & 1, m & 1
        a, b = small_frag(current, 0, ks, i), small_frag(current, 1, ks, j)
        lines.append("v_mfma_f32_32x32x16_bf16 %s, v[%d:%d], v[%d:%d], %s" % (
            SMALL_ACC(i, j), a, a + 3, b, b + 3, SMALL_ACC(i, j)))
        lines += behind[m]
    return lines


def small_loop(via=None, ring=4):
    lines = ["s_mov_b64 s[40:41], " + SMALL_IN["src_a"], "s_mov_b64 s[42:43], " + SMALL_IN["src_b"], "s_mov_b32 s44, %d" % ring]
    if via is not None:     # (the source of an operand through registers is that of step 0)
        first = SMALL_SETS[via][1]
        if via == 0:
            # steps 0 and 1, then as many as there are sets (steps 4 and 5 only if there are any)
            for k, registers in enumerate([first, first + 8] + [SMALL_VIA + 8 * ((k + 2) % (ring // 2)) for k in range(ring // 2)]):
                if k > 3:
                    lines += ["s_cmp_gt_u32 %s, 4" % SMALL_IN["steps"]] + small_names(ADVANCE_A[1:])
                elif k:
                    lines += ["s_add_u32 s40, s40, " + SMALL_IN["stride_a"], "s_addc_u32 s41, s41, 0"]
                lines += [small_load(0, n, registers) for n in range(2)]
        else:
            lines += [small_load(1, n, first) for n in range(4)] + ["s_add_u32 s42, s42, 128", "s_addc_u32 s43, s43, 0"]
            lines += [small_load(1, n, SMALL_VIA) for n in range(4)]
        # steps 0 and 1 and all copies have landed
        lines.append("s_waitcnt vmcnt(%d)" % ring)
        lines += [small_to_lds(1, n, first, 0) for n in range(4)] if via else [
            small_to_lds(0, n, first + 8 * k, k) for k in range(2) for n in range(2)]
        lines += ["s_waitcnt lgkmcnt(0)", "s_barrier"]
    lines += small_reads(0, SMALL_SETS[via][0])
    # (s44 has advanced with the steps; the last one read fragments that nobody uses)
    more = ["s_sub_u32 s45, s44, %d" % ring, "s_cmp_lt_u32 s45, " + SMALL_IN["steps"]]
    done = more + ["s_cbranch_scc0 ct_gemm_small_done_%="]

    def body(first_iteration=False):
        out = []
        for u in range(ring):
            behind_chunk = {4: {0: 3}, 8: {0: 7, 1: 7, 2: 11, 3: 11}}[ring].get(u) if first_iteration else None
            out += small_step(u, via, ring, behind_chunk) + (done if u == 3 and ring == 8 else [])
        return out

    if via is not None:
        lines += body(True) + done
    lines.append("ct_gemm_small_loop_%=:")
    lines += body() + more + ["s_cbranch_scc1 ct_gemm_small_loop_%="]
    if via is not None or ring == 8:
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
    print("#define CT_GEMM_LOOP_CLOBBERS %s" % clobbers(F0A, F1B + 16))
    print(emit(gemm_loop(fresh=True, via=0), "CT_GEMM_VIA_A_LOOP"))
    print(emit(gemm_loop(via=1), "CT_GEMM_VIA_B_LOOP"))
    print("#define CT_GEMM_VIA_LOOP_CLOBBERS %s" % clobbers(VIA, F1B + 16))
    print(emit(small_loop(), "CT_GEMM_SMALL_LOOP"))
    print("#define CT_GEMM_SMALL_LOOP_CLOBBERS %s" % clobbers(SMALL_SETS[None][0], SMALL_SETS[None][1] + 32))
    print(emit(small_loop(via=0), "CT_GEMM_SMALL_VIA_A_LOOP"))
    print(emit(small_loop(via=1), "CT_GEMM_SMALL_VIA_B_LOOP"))
    print("#define CT_GEMM_SMALL_VIA_LOOP_CLOBBERS %s" % clobbers(SMALL_SETS[0][0], SMALL_VIA + 16))
    print(emit(small_loop(ring=8), "CT_GEMM_SMALL_DEEP_LOOP"))
    print(emit(small_loop(via=0, ring=8), "CT_GEMM_SMALL_DEEP_VIA_A_LOOP"))
    print("#define CT_GEMM_SMALL_DEEP_VIA_LOOP_CLOBBERS %s" % clobbers(SMALL_SETS[0][0], SMALL_VIA + 32))
