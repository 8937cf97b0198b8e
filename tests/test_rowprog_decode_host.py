"""The interpreter's decoded form of a row program (rowprog_vm.h) against the program itself, both
executed on expressions instead of numbers: every store has to receive the same expression.  No GPU:
the library decodes on the host."""
import ctypes as C
import random

import pytest

from nabla_amd.backend import isa, lib

FLAT, ROW, LOOP = 0, 1, 2  # rp_vm_mode
(V_STG, V_STR, V_LD, V_LDG, V_LDS, V_LDR, V_COLIDX, V_RED, V_ACCINIT, V_ACC, V_IMM, V_LEADIDX, V_SEG) = range(1, 14)
SCALAR, NONE, ROW_SLOTS = 32, 255, 4
MAX_INS = isa.MAX_INS + isa.MAX_INS // 3 + 6


class VmIns(C.Structure):
    _fields_ = [(n, C.c_uint8) for n in ("op", "dst", "a", "b", "c", "two")] + [("aux", C.c_uint16)]


class Vm(C.Structure):
    _fields_ = [("lead_dim", C.c_int64 * isa.MAX_LEAD), ("C", C.c_int64), ("n_lead", C.c_int32),
                ("n_once", C.c_int32), ("n_ins", C.c_int32), ("n_slots", C.c_int32), ("n_row_slots", C.c_int32),
                ("lanes", C.c_int32), ("rare", C.c_int32), ("slots", C.c_uint8 * 44),
                ("row_slots", C.c_uint8 * ROW_SLOTS), ("row_dst", C.c_uint8 * ROW_SLOTS),
                ("imm", C.c_float * (isa.MAX_IMM + 1)), ("operand", lib.Operand * isa.MAX_OPERANDS),
                ("ins", VmIns * MAX_INS)]


def decode(rp, mode):
    """The decoded form, or None where ``mode`` does not take the program."""
    fn = getattr(lib.load(), "_Z12rp_vm_decodePK11nbk_rowprogiP5rp_vm")
    fn.restype, fn.argtypes = C.c_bool, [C.c_void_p, C.c_int, C.c_void_p]
    room = (C.c_uint8 * (C.sizeof(Vm) + 64))(*[0xA5] * (C.sizeof(Vm) + 64))
    vm = Vm.from_buffer(room)
    if not fn(C.byref(rp), mode, C.byref(vm)):
        return None
    assert bytes(room)[C.sizeof(Vm):] == b"\xa5" * 64 and 0 <= vm.n_once <= vm.n_ins <= MAX_INS
    return vm


_EXPRESSIONS: dict = {}


def E(*parts):
    """The number of an expression whose operands are numbers too (a value read twice is one)."""
    return _EXPRESSIONS.setdefault(parts, len(_EXPRESSIONS))


UNARY, TERNARY = set(isa.UNARY.values()), set(isa.TERNARY.values())


class Memory:
    """What loads yield and stores leave: expressions by operand and number of stores before."""

    def __init__(self):
        self.stores, self.version = [], {}

    def load(self, kind, operand):
        return E(kind, operand, self.version.get(operand, 0))

    def store(self, kind, operand, value):
        self.stores.append((kind, operand, value))
        self.version[operand] = self.version.get(operand, 0) + 1


def run_program(rp):
    """Stores of the program as nbk.h defines it."""
    mem, reg, acc = Memory(), {}, {}
    body = 0
    for i in range(rp.n_ins):
        n = rp.ins[i]
        if n.op == isa.HALT:
            break
        if n.op == isa.BODY:
            body = n.aux
            continue
        if n.op == isa.LDG:
            reg[n.dst] = mem.load("ldg", n.a)
        elif n.op == isa.LDR:
            reg[n.dst] = mem.load("ldr", n.a)
        elif n.op == isa.STG:
            mem.store("stg", n.dst, reg[n.a])
        elif n.op == isa.STR:
            mem.store("str", n.dst, reg[n.a])
        elif n.op == isa.IMM:
            reg[n.dst] = E("imm", n.a)
        elif n.op == isa.COLIDX:
            reg[n.dst] = E("col", int(n.a != 0))
        elif n.op == isa.LEADIDX:
            reg[n.dst] = E("lead", n.a, int(n.b != 0))
        elif n.op == isa.ACCINIT:
            acc[n.dst] = (("init", n.a),)
        elif n.op == isa.ACC:
            acc[n.dst] = acc[n.dst] + (("acc", n.b, reg[n.a]),)
        elif n.op == isa.RED:
            reg[n.dst] = E("red", n.b, acc[n.a])
        else:
            args = (n.a,) if n.op in UNARY else (n.a, n.b, n.c) if n.op in TERNARY else (n.a, n.b)
            reg[n.dst] = E(n.op, *(reg[r] for r in args))
        body -= 1
    return mem.stores


def run_decoded(vm, mode, wave=True):
    """Stores of the decoded form as rp_vm_kernel executes it; ``wave``: a row held by one wavefront
    (grouped reductions then write their scalars from the last to the first)."""
    mem, vec, scl, acc = Memory(), {}, {}, {}

    def get(r):
        return scl[r - SCALAR] if r >= SCALAR else vec[r]

    def put(dst, value):
        if dst < isa.NVEC:
            vec[dst] = value
        elif dst != NONE:
            assert SCALAR <= dst < SCALAR + isa.NSCL
            scl[dst - SCALAR] = value

    for k in range(vm.n_row_slots):
        put(vm.row_dst[k], mem.load("ldr", vm.row_slots[k]))

    def segment(q0, q1):
        q = q0
        while q < q1:
            n = vm.ins[q]
            if n.op == V_RED:
                group = [vm.ins[q + k] for k in range(n.aux)]
                assert all(m.op == V_RED for m in group) and 1 <= n.aux <= 4
                if mode == LOOP:
                    value = lambda m: E("red", m.b, acc[m.c])
                else:
                    value = lambda m: E("red", m.b, (("init", m.b), ("acc", m.b, get(m.a))))
                if wave:
                    for m in reversed(group):
                        put(m.dst, value(m))
                else:
                    for m, v in [(m, value(m)) for m in group]:
                        put(m.dst, v)
                q += n.aux
                continue
            if n.op >= isa.UNARY["mov"]:
                args = (n.a, n.b, n.c) if n.op in TERNARY else (n.a, n.b) if n.two else (n.a,)
                put(n.dst, E(n.op, *(get(r) for r in args)))
            elif n.op in (V_LDG, V_LDR):
                put(n.dst, mem.load("ldg" if n.op == V_LDG else "ldr", n.c))
            elif n.op in (V_STG, V_STR):
                mem.store("stg" if n.op == V_STG else "str", n.c, get(n.a))
            elif n.op == V_COLIDX:
                put(n.dst, E("col", int(n.c != 0)))
            elif n.op == V_IMM:
                put(n.dst, E("imm", n.c))
            elif n.op == V_LEADIDX:
                put(n.dst, E("lead", n.c, int(n.b != 0)))
            elif n.op == V_ACCINIT:
                acc[n.c] = (("init", n.b),)
            elif n.op == V_ACC:
                acc[n.c] = acc[n.c] + (("acc", n.b, get(n.a)),)
            else:
                raise AssertionError(n.op)
            q += 1

    if mode != LOOP:
        for k in range(vm.n_slots):
            vec[k] = mem.load("ldg", vm.slots[k])
        segment(0, vm.n_ins)
        return mem.stores
    q1 = 0
    while q1 < vm.n_ins:
        seg = vm.ins[q1]
        assert seg.op == V_SEG
        q0, q1 = q1 + 1, q1 + 1 + seg.aux
        vec.clear()  # (a chunk's registers do not outlive its segment)
        for k in range(seg.a):
            vec[k] = mem.load("ldg", vm.slots[seg.c + k])
        segment(q0, q1)
    return mem.stores


def program(ins, n_operands, cols, reduce, moves=()):
    """A launch record over rows of ``cols`` floats; operands ``moves`` change with the row."""
    rp = lib.RowProg()
    rp.n_lead, rp.lead_dim[0], rp.C, rp.block = 1, 7, cols, 256
    rp.n_operands, rp.n_imm, rp.has_reduce = n_operands, isa.MAX_IMM, int(reduce)
    for i in range(n_operands):
        rp.operand[i].ptr, rp.operand[i].col_stride, rp.operand[i].stage_slot = 4096, 1, -1
        rp.operand[i].lead_stride[0] = cols if i in moves else 0
    for i in range(isa.MAX_IMM):
        rp.imm[i] = i - isa.MAX_IMM // 2
    ins = ins + [(isa.HALT, 0, 0, 0, 0, 0)]
    assert len(ins) <= isa.MAX_INS
    rp.n_ins = len(ins)
    for i, n in enumerate(ins):
        d = rp.ins[i]
        d.op, d.dst, d.a, d.b, d.c, d.aux = n
    return rp


def check(rp):
    """Decodes and compares every mode that a launch may use; what each made of the program."""
    want = run_program(rp)
    modes = [ROW, LOOP] if rp.has_reduce else [FLAT]
    forms = {m: decode(rp, m) for m in modes}
    for m, vm in forms.items():
        if vm is not None:
            assert run_decoded(vm, m) == want, m
            assert run_decoded(vm, m, wave=False) == want, m
    # (rows that no register file holds are walked in chunks: that form takes any program)
    assert forms[modes[-1]] is not None
    return forms


def body(*ins):
    return [(isa.BODY, 0, 0, 0, 0, len(ins)), *ins]


def shared_inputs_program(rng):
    """Two or three phases over the same inputs, each reading all of them in an order of its own,
    with more values than registers to keep them in until the next phase."""
    n_in = rng.randint(3, 10)
    ins = []
    for phase in range(rng.randint(2, 3)):
        ins.append((isa.ACCINIT, phase, 1, 0, 0, 0))
        b, free = [], list(range(isa.NVEC))
        held, total, cond = {}, free.pop(), []
        order = rng.sample(range(n_in), n_in)
        for k, i in enumerate(order):
            held[i] = free.pop()
            b.append((isa.LDG, held[i], i, 0, 0, 0))
            if k == 0:
                b.append((isa.UNARY["neg"], total, held[i], 0, 0, 0))
            elif len(free) > n_in - 1 - k:
                cond.append(free.pop())
                b.append((isa.BINARY["gt"], cond[-1], held[i], held[order[k - 1]], 0, 0))
                b.append((isa.TERNARY["where"], total, cond[-1], held[i], total, 0))
            if rng.random() < 0.3 and phase:
                b.append((isa.BINARY["sub"], held[i], held[i], isa.NVEC, 0, 0))
        rng.shuffle(cond)
        for c in cond:
            b.append((isa.BINARY["mul"], total, total, c, 0, 0))
        b += [(isa.ACC, phase, total, 1, 0, 0), (isa.STG, n_in + phase, total, 0, 0, 0)]
        ins += body(*b) + [(isa.RED, isa.NVEC, phase, 1, 0, 0)]
    return program(ins, n_in + 3, rng.choice([1, 100, 1003]), True, range(n_in + 3))


def inputs_and_stores(rp):
    """Operands that the program loads, and those that it stores."""
    loads, stores = set(), set()
    for i in range(rp.n_ins):
        n = rp.ins[i]
        if n.op in (isa.LDG, isa.LDR):
            loads.add(n.a)
        elif n.op in (isa.STG, isa.STR):
            stores.add(n.dst)
    return loads, stores


def random_program(rng, exact=False):
    """A valid program: bodies that read what they or the prologues wrote, reductions between
    them, inputs read again, row scalars loaded twice, all registers in use.  ``exact``: operations that
    keep whole numbers, no integer registers, and outputs that are only written."""
    reduce, once = rng.random() < 0.75, rng.random() < 0.7  # (once: accumulators that rows in registers can have)
    n_in, n_out = rng.randint(1, 14), rng.randint(1, 5)
    n_vec, n_scl = rng.choice([4, 8, 12, 16, 16]), rng.choice([3, 8, 16])
    moves = [i for i in range(n_in + n_out) if rng.random() < 0.7 or exact and i >= n_in]
    ops1 = [isa.UNARY[k] for k in ("neg", "abs" if exact else "exp", "relu")]
    ops2 = [isa.BINARY[k] for k in (("gt", "sub", "gt") if exact else ("add", "sub", "mul", "gt"))]
    scalars, ins, started = [], [], {}

    def ew(regs, dst):
        kind = rng.random()
        if kind < 0.25:
            return (rng.choice(ops1), dst, rng.choice(regs), 0, 0, 0)
        if kind < 0.8:
            return (rng.choice(ops2), dst, rng.choice(regs), rng.choice(regs), 0, 0)
        return (isa.TERNARY["where"] if exact else rng.choice(sorted(TERNARY)), dst, *(rng.choice(regs) for _ in range(3)), 0)

    for _ in range(rng.randint(1, 4)):
        for _ in range(rng.randint(0, 2 + n_scl // 2)):
            dst = isa.NVEC + rng.randrange(n_scl)
            kind = rng.random()
            if kind < 0.4:
                ins.append((isa.LDR, dst, rng.randrange(n_in), 0, 0, 0))
            elif kind < 0.6 or not scalars:
                ins.append((isa.IMM, dst, rng.randrange(isa.MAX_IMM), 0, 0, 0))
            elif kind < 0.7:
                ins.append((isa.LEADIDX, dst, 0, 0 if exact else rng.randint(0, 1), 0, 0))
            elif kind < 0.75:
                ins.append((isa.STR, n_in + rng.randrange(n_out), rng.choice(scalars), 0, 0, 0))
                continue
            else:
                ins.append(ew(scalars, dst))
            scalars.append(dst) if dst not in scalars else None
        if reduce:
            for k in range(isa.NACC):
                if rng.random() < 0.6 and not (once and started.get(k, (0, 0))[1]):
                    kind = rng.randrange(1 if exact else 0, 3)
                    ins.append((isa.ACCINIT, k, kind, 0, 0, 0))
                    started[k] = [kind, 0]
        vecs, b = [], []
        for _ in range(rng.randint(2, 30)):
            dst = rng.randrange(n_vec)
            kind = rng.random()
            if kind < 0.4 or not vecs:
                b.append((isa.LDG, dst, rng.randrange(n_in + (n_out if rng.random() < 0.1 and not exact else 0)), 0, 0, 0))
            elif kind < 0.43:
                b.append((isa.COLIDX, dst, 0 if exact else rng.randint(0, 1), 0, 0, 0))
            elif kind < 0.5:
                b.append((isa.STG, n_in + rng.randrange(n_out), rng.choice(vecs + scalars), 0, 0, 0))
                continue
            elif kind < 0.6 and any(n == 0 or not once for _, n in started.values()):
                k = rng.choice([k for k in sorted(started) if started[k][1] == 0 or not once])
                b.append((isa.ACC, k, rng.choice(vecs + vecs + scalars), started[k][0], 0, 0))
                started[k][1] += 1
                continue
            else:
                b.append(ew(vecs + scalars, dst))
            if dst not in vecs:
                vecs.append(dst)
        b.append((isa.STG, n_in + rng.randrange(n_out), rng.choice(vecs), 0, 0, 0))
        ins += body(*b)
        for k in sorted(started):
            if started[k][1] and rng.random() < 0.8:
                # (a second reduction of the same accumulator too, in a later phase)
                dst = isa.NVEC + rng.randrange(n_scl)
                ins.append((isa.RED, dst, k, started[k][0], 0, 0))
                if dst not in scalars:
                    scalars.append(dst)
    ins += body((isa.LDG, 0, 0, 0, 0, 0), *[(isa.BINARY["add"], 0, 0, s, 0, 0) for s in scalars],
                (isa.STG, n_in, 0, 0, 0, 0))
    return program(ins, n_in + n_out, rng.choice([1, 3, 100, 1003, 5000]), reduce, moves)


@pytest.mark.parametrize("seed", range(8))
def test_random_programs(seed):
    rng = random.Random(seed)
    for _ in range(250):
        check(random_program(rng))


@pytest.mark.parametrize("seed", range(4))
def test_inputs_read_again_in_a_later_phase(seed):
    rng = random.Random(seed)
    held = [check(shared_inputs_program(rng))[ROW] is not None for _ in range(150)]
    assert sum(held) > 75  # (rows in registers, the form that requests an input once for all phases)


def test_all_scalars_alive_and_row_operands_loaded_twice():
    """Sixteen scalars that every phase reads, the operands of a row among them, loaded again into
    registers that are needed in between."""
    rng = random.Random(1)
    for n_row in range(1, 17):
        S = isa.NVEC
        ins = [(isa.LDR, S + k, k % n_row, 0, 0, 0) for k in range(16)]
        for phase in range(3):
            order = rng.sample(range(16), 16)
            ins += [(isa.ACCINIT, 0, 0, 0, 0, 0)]
            ins += body((isa.LDG, 0, 16, 0, 0, 0), *[(isa.BINARY["mul"], 0, 0, S + k, 0, 0) for k in order],
                        (isa.ACC, 0, 0, 0, 0, 0), (isa.STG, 17, 0, 0, 0, 0))
            ins += [(isa.RED, S + order[0], 0, 0, 0, 0)]
            ins += [(isa.BINARY["add"], S + order[k], S + order[k], S + order[k - 1], 0, 0) for k in (1, 2)]
            ins += [(isa.LDR, S + order[k], order[k] % n_row, 0, 0, 0) for k in (3, 4)]
        check(program(ins, 18, 1003, True, range(18)))


def test_the_longest_programs():
    """As many instructions as a record holds, in the pattern whose looped form grows the most: a
    scalar behind every body."""
    for reduce in (False, True):
        S = isa.NVEC
        ins = [(isa.LDR, S + k, 0, 0, 0, 0) for k in range(1)]
        while len(ins) + 4 <= isa.MAX_INS:
            ins += body((isa.STG, 1, S, 0, 0, 0)) + [(isa.BINARY["add"], S, S, S, 0, 0)]
        check(program(ins, 2, 100, reduce, [0, 1]))


@pytest.mark.parametrize("kinds", [(1, 0), (0, 0, 0), (2, 1, 0, 1)])
def test_a_reduction_of_its_neighbours_result(kinds):
    """Nothing but bodies stands between the reductions, and a body leaves nothing behind."""
    S = isa.NVEC
    ins = [(isa.ACCINIT, k, kind, 0, 0, 0) for k, kind in enumerate(kinds)]
    ins += body((isa.LDG, 0, 0, 0, 0, 0), (isa.ACC, 0, 0, kinds[0], 0, 0)) + [(isa.RED, S, 0, kinds[0], 0, 0)]
    for k in range(1, len(kinds)):
        ins += body((isa.ACC, k, S + (k - 1) % 2, kinds[k], 0, 0)) + [(isa.RED, S + k % 2, k, kinds[k], 0, 0)]
    last = S + (len(kinds) - 1) % 2
    ins += body((isa.STG, 1, last, 0, 0, 0))
    assert check(program(ins, 2, 1003, True, [0, 1]))[ROW] is not None


def test_instructions_of_scalars_name_scalars_only():
    """All three operands are read, whatever the instruction has: a register number below the scalars would be
    an index outside their file."""
    rng, seen = random.Random(5), 0
    for _ in range(200):
        rp = random_program(rng)
        for mode in [ROW, LOOP] if rp.has_reduce else [FLAT]:
            vm = decode(rp, mode)
            for q in range(vm.n_ins if vm is not None else 0):
                n = vm.ins[q]
                if n.op >= isa.UNARY["mov"] and SCALAR <= n.dst < NONE:
                    assert all(SCALAR <= r < SCALAR + isa.NSCL for r in (n.a, n.b, n.c)), (n.op, n.a, n.b, n.c)
                    seen += 1
    assert seen > 200
