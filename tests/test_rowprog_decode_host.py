"""The interpreter's decoded form of a row program (rowprog_vm.h) against the program itself, both
executed on expressions instead of numbers: every store has to receive the same expression.  No GPU:
the library decodes on the host."""
import ctypes as C
import random
import re

import pytest

from nabla_amd.backend import isa, lib

FLAT, ROW, LOOP = 0, 1, 2  # rp_vm_mode
(V_STG, V_STR, V_LD, V_LDG, V_LDS, V_LDR, V_COLIDX, V_RED, V_ACCINIT, V_ACC, V_IMM, V_LEADIDX, V_SEG) = range(1, 14)
SCALAR, NONE, ROW_SLOTS = 32, 255, 4
MAX_INS = int(re.search(r"RPVM_MAX_INS (\d+)", (lib.LIB_PATH.parent / "rowprog_vm.h").read_text())[1])


class VmIns(C.Structure):
    _fields_ = [(n, C.c_uint8) for n in ("op", "dst", "a", "b", "c", "two")] + [("aux", C.c_uint16)]


class Vm(C.Structure):
    _fields_ = [("lead_dim", C.c_int64 * isa.MAX_LEAD), ("C", C.c_int64), ("n_lead", C.c_int32),
                ("n_once", C.c_int32), ("n_ins", C.c_int32), ("n_slots", C.c_int32), ("n_row_slots", C.c_int32),
                ("lanes", C.c_int32), ("file", C.c_int16), ("rare", C.c_int16), ("slots", C.c_uint8 * 44),
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
        if dst < vm.file:
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


@pytest.mark.parametrize("seed", range(4))
def test_inputs_read_again_in_a_later_phase(seed):
    rng = random.Random(seed)
    held = [check(shared_inputs_program(rng))[ROW] is not None for _ in range(150)]
    assert sum(held) > 75  # (rows in registers, the form that requests an input once for all phases)
