"""The main loops that gen_gemm_asm.py emits, run on a model of one wavefront.

The loops count their copies and LDS reads in flight themselves, so a wait that is too weak is a race on LDS that no GPU
test reliably shows. In the model copies and stores complete in the order of their issue and no sooner than a wait asks for;
the four wavefronts of a workgroup run the same stream, so what one of them has waited for before a barrier, all have.
Checked for every instruction: an LDS read finds the copies of its step landed in front of a barrier, a copy goes where
every read is done in front of a barrier and no other copy is on its way, and every MFMA has the fragments of its step.
An operand that comes through registers: a chunk's load has landed when it is stored to LDS, and the store counts as a copy
that has landed once the wavefront has waited for it.
"""

import importlib.util
import os
import re
import subprocess
import sys

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "causal-trainer-dev_amd", "csrc")
GENERATOR = os.path.join(CSRC, "gen_gemm_asm.py")


@pytest.fixture(scope="module")
def gen():
    spec = importlib.util.spec_from_file_location("gen_gemm_asm", GENERATOR)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


class Tile:
    """What the operands of a loop's asm statement stand for, and the layout of its LDS stages: `ring` (four, or eight in
    the small tile) of A, a step each, then half as many of B, a pair of steps each."""

    def __init__(self, small, ring=4):
        self.blocks = 2 if small else 4                     # of a wavefront, in each direction
        self.chunks = (self.blocks, 2 * self.blocks)        # copies of a wavefront per stage
        # stages copied in front of the loop
        self.ahead = ((0, 0), (1, 0), (0, 1), (1, 1), (0, 2), (0, 3)) if small else ((0, 0), (1, 0), (0, 1), (0, 2), (1, 1))
        if ring == 8:
            self.ahead = ((0, 0), (1, 0), (0, 1), (0, 2), (1, 1), (0, 3), (0, 4), (1, 2), (0, 5), (0, 6), (1, 3), (0, 7))
        self.ring, self.a_stage = ring, 8192 if small else 16384
        self.b_at, self.b_stage = ring * self.a_stage, 2 * self.a_stage
        first = self.blocks ** 2                            # (the accumulators are operands 0 ..)
        self.src = {"%%%d" % first: 0, "%%%d" % (first + 1): 1}
        self.stride, self.steps, self.lds_wave = ("%%%d" % (first + k) for k in (2, 3, 4))
        self.reads, self.copies = {}, {}                    # operand -> (matrix, second, block or k-step of a pair), (matrix, chunk)
        at = first + 5
        for second in range(2):
            for block in range(self.blocks):
                self.reads["%%%d" % at] = (0, second, block)
                at += 1
        for ks in range(4):
            self.reads["%%%d" % at] = (1, None, ks)
            at += 1
        for matrix in range(2):
            for chunk in range(self.chunks[matrix]):
                self.copies["%%%d" % at] = (matrix, chunk)
                at += 1
        self.thread = "%%%d" % at

    def place(self, offset):
        """(matrix, stage, chunk) of 4 KB of LDS"""
        matrix = int(offset >= self.b_at)
        stage, rest = divmod(offset - matrix * self.b_at, self.b_stage if matrix else self.a_stage)
        chunk, rest = divmod(rest, 4096)
        assert rest == 0 and stage < (self.ring // 2 if matrix else self.ring)
        return matrix, stage, chunk


class Machine:
    """One wavefront on a loop of `steps` steps. `stores` lie behind the copies of the first steps; `start_wait`: the
    vmcnt in front of the loop; `via`: the operand that comes through registers."""

    # bytes from step to step of the two sources (the first carries into the upper half of the address), and between them
    STRIDE, HIGH = ((1 << 32) - 4096, 64), 1 << 40
    # (a slot's step: A's, or the first of B's pair)

    def __init__(self, tile, steps, fresh, stores, start_wait, via=None):
        self.tile, self.steps, self.fresh, self.via = tile, steps, fresh, via
        self.scalar, self.scc, self.fragment = {}, 0, {}
        self.loaded, self.lds_stores = {}, []               # first register -> what a load puts there; on their way to LDS
        self.memory, self.lds_reads = [], []                # in flight, in the order of their issue
        self.slots, self.mfmas, self.started = {}, 0, set()
        # (in the order of ct_gemm.hip.h)
        for matrix, stage in tile.ahead:
            for chunk in range(tile.chunks[matrix]):
                if matrix != via:                           # (past the end the last step's again, which nobody reads)
                    self._copy(matrix, chunk, stage * (1 + matrix), stage)
        self.memory += [None] * stores
        if start_wait is not None:
            self._wait_memory(start_wait)
            self._barrier()

    # -- events
    def _copy(self, matrix, chunk, step, stage, flight=None):
        slot = self.slots.setdefault((stage, matrix, chunk), dict(state="free", readers=[]))
        assert slot["state"] != "flying", ("a copy on its way to the same place", stage, matrix, chunk)
        assert all(reader == "fenced" for reader in slot["readers"]), ("a copy over data being read", stage, matrix, chunk)
        slot.update(state="flying", step=step, readers=[])
        (self.memory if flight is None else flight).append(slot)

    def _load(self, matrix, chunk, step, registers):
        assert matrix == self.via
        for register in registers:
            assert self.fragment.get(register, [None, True])[1], ("load into a register of a read in flight", register)
            self.fragment.pop(register, None)
        held = self.loaded[registers[0]] = dict(state="flying", matrix=matrix, chunk=chunk, step=step)
        self.memory.append(held)

    def _store(self, registers, where, offset):
        assert where == self.tile.thread
        held = self.loaded[registers[0]]
        assert held["state"] == "landed", ("store of a chunk that has not landed", held)
        matrix, stage, chunk = self.tile.place(offset + self.via * self.tile.b_at)
        assert (matrix, chunk) == (held["matrix"], held["chunk"])
        self._copy(matrix, chunk, held["step"], stage, self.lds_stores)

    def _wait_memory(self, most):
        assert most <= 63
        while len(self.memory) > most:
            slot = self.memory.pop(0)
            if slot is not None:
                slot["state"] = "landed"

    def _wait_lds(self):
        for slot in self.lds_stores:
            slot["state"] = "landed"
        self.lds_stores = []
        for slots, registers in self.lds_reads:
            for slot, index in slots:
                slot["readers"][index] = "done"
            for register in registers:
                self.fragment[register][1] = True
        self.lds_reads = []

    def _barrier(self):
        for slot in self.slots.values():
            if slot["state"] == "landed":
                slot["state"] = "there"
            slot["readers"] = ["fenced" if reader in ("done", "fenced") else reader for reader in slot["readers"]]

    def _read(self, registers, operand, offset):
        matrix, second, which = self.tile.reads[operand]
        if matrix == 0:                                     # rows of the contraction: half of the tile per k-step
            stage, rest = divmod(offset, self.tile.a_stage)
            ks, rest = divmod(rest, self.tile.a_stage // 2)
            half = self.tile.chunks[0] // 2
            block, parity, chunks = which, 0, range(ks * half, (ks + 1) * half)
        else:
            stage, rest = divmod(offset, self.tile.b_stage)
            block, rest = divmod(rest, 4096)
            parity, ks = divmod(which, 2)
            chunks = range(self.tile.chunks[1])             # (half of them, by the wavefront)
        assert rest == 0 and block < self.tile.blocks, operand
        slots = []
        for chunk in chunks:
            assert (stage, matrix, chunk) in self.slots, ("LDS read of a place that nothing was copied to", stage, matrix, chunk)
            slot = self.slots[stage, matrix, chunk]
            assert slot["state"] == "there", ("LDS read ahead of its copies", stage, matrix, chunk, slot["state"])
            slot["readers"].append("pending")
            slots.append((slot, len(slot["readers"]) - 1))
        assert not any(register in range(first, first + 4) and held["state"] == "flying"
                       for first, held in self.loaded.items() for register in registers)
        step = slots[0][0]["step"]
        assert all(slot["step"] == step for slot, _ in slots)
        step += parity
        for k, register in enumerate(registers):
            assert self.fragment.get(register, [None, True])[1], ("register of a read in flight", register)
            self.fragment[register] = [(matrix, step, ks, block, second if matrix == 0 else k // 2), False]
        self.lds_reads.append((slots, registers))
        assert len(self.lds_reads) <= 15

    def _mfma(self, d, a, b, c):
        blocks = self.tile.blocks
        per_step = 2 * blocks ** 2
        step, (ks, (i, j)) = self.mfmas // per_step, (self.mfmas % per_step // blocks ** 2, divmod(self.mfmas % blocks ** 2, blocks))
        assert d == "%%%d" % (blocks * i + j)
        for matrix, block, operand in ((0, i, a), (1, j, b)):
            for k, register in enumerate(_registers(operand)):
                assert self.fragment[register] == [(matrix, step, ks, block, k // 2), True], (step, d, operand, self.fragment[register])
        if self.fresh and d not in self.started:
            assert c == "0"
        else:
            assert c == d
        self.started.add(d)
        self.mfmas += 1

    # -- scalar instructions
    def _get(self, operand):
        if operand in self.tile.src:                        # address of the copies of step 3
            matrix = self.tile.src[operand]
            ring = self.tile.ring
            step = 0 if matrix == self.via else min(ring, self.steps - 2) if matrix else min(ring, self.steps) - 1
            return matrix * self.HIGH + step * self.STRIDE[matrix]
        if operand == self.tile.stride:
            return self.STRIDE[0]
        if operand == self.tile.steps:
            return self.steps
        if operand == self.tile.lds_wave:
            return 0
        if operand.startswith(("s", "m0")):
            return self.scalar[operand]
        return int(operand, 0)

    def run(self, lines):
        labels = {line[:-1]: at for at, line in enumerate(lines) if line.endswith(":")}
        at = executed = 0
        while at < len(lines):
            line = lines[at]
            at += 1
            executed += 1
            assert executed < 100000
            if line.endswith(":"):
                continue
            name, _, rest = line.partition(" ")
            ops = [part.strip() for part in rest.split(",")]
            if name == "s_waitcnt":
                counter, most = re.fullmatch(r"(vmcnt|lgkmcnt)\((\d+)\)", rest).groups()
                if counter == "vmcnt":
                    self._wait_memory(int(most))
                else:
                    assert int(most) == 0
                    self._wait_lds()
            elif name == "s_barrier":
                self._barrier()
            elif name.startswith("ds_read"):
                where, _, offset = ops[1].partition(" offset:")
                self._read(_registers(ops[0]), where, int(offset))
            elif name == "ds_write_b128":
                registers, _, offset = ops[1].partition(" offset:")
                self._store(_registers(registers), ops[0], int(offset))
            elif name in ("global_load_lds_dwordx4", "global_load_dwordx4"):
                target = ops.pop(0) if name == "global_load_dwordx4" else None
                matrix, chunk = self.tile.copies[ops[0]]
                low = int(re.fullmatch(r"s\[(\d+):\d+\]", ops[1]).group(1))
                source = (self.scalar["s%d" % (low + 1)] << 32 | self.scalar["s%d" % low]) - matrix * self.HIGH
                step, rest = divmod(source, self.STRIDE[matrix])
                assert rest == 0 and 0 <= step < self.steps, ("copy from outside of the matrix", step)
                assert matrix == 0 or step % 2 == 0, ("half of a pair", step)
                if target is not None:
                    self._load(matrix, chunk, step, _registers(target))
                    continue
                place = self.tile.place(self.scalar["m0"])
                assert (place[0], place[2]) == (matrix, chunk)
                self._copy(matrix, chunk, step, place[1])
            elif name == "v_mfma_f32_32x32x16_bf16":
                self._mfma(*ops)
            elif name == "s_mov_b64":
                low, high = re.fullmatch(r"s\[(\d+):(\d+)\]", ops[0]).groups()
                value = self._get(ops[1])
                self.scalar["s" + low], self.scalar["s" + high] = value & 0xffffffff, value >> 32
            elif name == "s_mov_b32":
                self.scalar[ops[0]] = self._get(ops[1])
            elif name in ("s_add_u32", "s_addc_u32"):
                value = self._get(ops[1]) + self._get(ops[2]) + (self.scc if name == "s_addc_u32" else 0)
                self.scalar[ops[0]], self.scc = value & 0xffffffff, value >> 32
            elif name == "s_sub_u32":
                value = self._get(ops[1]) - self._get(ops[2])
                self.scalar[ops[0]], self.scc = value & 0xffffffff, int(value < 0)
            elif name == "s_cmp_lt_u32":
                self.scc = int(self._get(ops[0]) < self._get(ops[1]))
            elif name == "s_cmp_gt_u32":
                self.scc = int(self._get(ops[0]) > self._get(ops[1]))
            elif name == "s_cselect_b32":
                self.scalar[ops[0]] = self._get(ops[1] if self.scc else ops[2])
            elif name in ("s_cbranch_scc0", "s_cbranch_scc1"):
                if self.scc == int(name[-1]):
                    at = labels[rest]
            else:
                assert name == "s_nop", line
        assert self.mfmas == self.steps * 2 * self.tile.blocks ** 2
        assert not self.memory and not self.lds_reads and not self.lds_stores
        # the next tile's copies may go anywhere
        assert all(reader == "fenced" for slot in self.slots.values() for reader in slot["readers"])


def _registers(operand):
    low, high = re.fullmatch(r"v\[(\d+):(\d+)\]", operand).groups()
    return range(int(low), int(high) + 1)


# loop -> (small tile, from C = 0, vmcnt in front of it, stores that may lie behind the first copies; as in ct_gemm.hip.h)
LOOPS = {"CT_GEMM_LOOP": (False, False, 16, (0,)), "CT_GEMM_FRESH_LOOP": (False, True, 16, (0,)),
         "CT_GEMM_FRESH_LOOP_BEHIND_STORES": (False, True, 63, (55, 64, 300)), "CT_GEMM_SMALL_LOOP": (True, False, 8, (0,)),
         "CT_GEMM_VIA_A_LOOP": (False, True, None, (0, 70)), "CT_GEMM_VIA_B_LOOP": (False, False, None, (0,)),
         "CT_GEMM_SMALL_VIA_A_LOOP": (True, False, None, (0, 70)), "CT_GEMM_SMALL_VIA_B_LOOP": (True, False, None, (0,))}
RING = {"CT_GEMM_SMALL_DEEP_LOOP": 8, "CT_GEMM_SMALL_DEEP_VIA_A_LOOP": 8}
LOOPS.update({"CT_GEMM_SMALL_DEEP_LOOP": (True, False, 26, (0,)), "CT_GEMM_SMALL_DEEP_VIA_A_LOOP": (True, False, None, (0, 70))})
VIA = {"CT_GEMM_SMALL_DEEP_VIA_A_LOOP": 0, "CT_GEMM_VIA_A_LOOP": 0, "CT_GEMM_VIA_B_LOOP": 1, "CT_GEMM_SMALL_VIA_A_LOOP": 0, "CT_GEMM_SMALL_VIA_B_LOOP": 1}


def _lines(gen, name):
    return {"CT_GEMM_LOOP": lambda: gen.gemm_loop(), "CT_GEMM_FRESH_LOOP": lambda: gen.gemm_loop(fresh=True),
            "CT_GEMM_FRESH_LOOP_BEHIND_STORES": lambda: gen.gemm_loop(fresh=True, behind_stores=True),
            "CT_GEMM_SMALL_LOOP": lambda: gen.small_loop(), "CT_GEMM_VIA_A_LOOP": lambda: gen.gemm_loop(fresh=True, via=0),
            "CT_GEMM_VIA_B_LOOP": lambda: gen.gemm_loop(via=1), "CT_GEMM_SMALL_VIA_A_LOOP": lambda: gen.small_loop(via=0),
            "CT_GEMM_SMALL_VIA_B_LOOP": lambda: gen.small_loop(via=1),
            "CT_GEMM_SMALL_DEEP_LOOP": lambda: gen.small_loop(ring=8),
            "CT_GEMM_SMALL_DEEP_VIA_A_LOOP": lambda: gen.small_loop(via=0, ring=8)}[name]()


def _run(lines, name, steps, stores, start_wait=None):
    small, fresh, wait, _ = LOOPS[name]
    machine = Machine(Tile(small, RING.get(name, 4)), steps, fresh, stores, wait if start_wait is None else start_wait, VIA.get(name))
    machine.run(lines)


@pytest.mark.parametrize("name", LOOPS)
def test_waits_and_fragments(gen, name):
    lines = _lines(gen, name)
    for steps in (4, 8, 12, 16, 20):
        for stores in LOOPS[name][3]:
            _run(lines, name, steps, stores)


def test_copies_that_have_landed_need_no_stores(gen):
    """A kernel's first tile, and one behind an epilogue with too few stores, wait for all copies in front of the loop."""

    for stores in (0, 7, 54):
        _run(_lines(gen, "CT_GEMM_FRESH_LOOP_BEHIND_STORES"), "CT_GEMM_FRESH_LOOP_BEHIND_STORES", 8, stores, start_wait=0)


def test_fewest_stores_are_what_the_header_waits_by(gen):
    with open(os.path.join(CSRC, "ct_gemm.hip.h")) as handle:
        fewest = int(re.search(r"kStoresBehindCopies = (\d+);", handle.read()).group(1))
    lines = _lines(gen, "CT_GEMM_FRESH_LOOP_BEHIND_STORES")
    _run(lines, "CT_GEMM_FRESH_LOOP_BEHIND_STORES", 8, fewest)
    with pytest.raises(AssertionError, match="LDS read ahead of its copies"):
        _run(lines, "CT_GEMM_FRESH_LOOP_BEHIND_STORES", 8, fewest - 1)


@pytest.mark.parametrize("name", LOOPS)
def test_model_catches_the_mistakes_it_is_meant_for(gen, name):
    stores = LOOPS[name][3][0]
    good = _lines(gen, name)

    def broken(change):
        lines = list(good)
        change(lines)
        with pytest.raises(AssertionError):
            _run(lines, name, 3 * RING.get(name, 4), stores)

    # every wait for copies, one copy weaker (63 is the largest there is)
    loop = next(at for at, line in enumerate(good) if "_loop_" in line)
    fragments = next(at for at, line in enumerate(good) if line.startswith("ds_read"))

    def binds(at):      # (the first iteration of an operand through registers finds the other's first copies landed)
        return name not in VIA or not fragments < at < loop or good[at + 1].startswith("ds_write")

    for at, line in enumerate(good):
        counted = re.fullmatch(r"s_waitcnt vmcnt\((\d+)\)", line)
        if counted and 0 < int(counted.group(1)) < 63 and binds(at):
            broken(lambda lines: lines.__setitem__(at, "s_waitcnt vmcnt(%d)" % (int(counted.group(1)) + 1)))
    # every barrier and every wait for LDS reads in front of the last ones gone
    for at, line in enumerate(good[:-6]):
        if line in ("s_barrier", "s_waitcnt lgkmcnt(0)") and binds(at):
            broken(lambda lines: lines.__setitem__(at, "s_nop 0"))
    # a fragment read from the next stage, and a copy to it
    tile = Tile(LOOPS[name][0], RING.get(name, 4))
    first = next(at for at, line in enumerate(good) if line.startswith("ds_read") and line.endswith("offset:0"))
    broken(lambda lines: lines.__setitem__(first, good[first].replace("offset:0", "offset:%d" % tile.a_stage)))
    copy = next(at for at, line in enumerate(good) if line.startswith("s_add_u32 m0"))
    operand, offset = re.fullmatch(r"s_add_u32 m0, (\S+), (\d+)", good[copy]).groups()
    other = (int(offset) + tile.a_stage) % tile.b_at if int(offset) < tile.b_at else (int(offset) - tile.b_at) ^ tile.b_stage
    broken(lambda lines: lines.__setitem__(copy, "s_add_u32 m0, %s, %d" % (operand, other)))
    # a source that moves on past the last step
    for chosen in dict.fromkeys(line for line in good if line.startswith("s_cselect_b32")):
        broken(lambda lines: [lines.__setitem__(at, chosen[:-1] + chosen.split(", ")[1]) for at, line in enumerate(good) if line == chosen])


def test_committed_include_is_what_the_generator_prints():
    printed = subprocess.run([sys.executable, GENERATOR], capture_output=True, text=True, check=True).stdout
    with open(os.path.join(CSRC, "ct_gemm_asm.inc")) as handle:
        assert handle.read() == printed
