"""Row programs whose inputs are read again in a later phase, with more values alive than the
interpreter's registers hold: results are comparisons and selections, exact in float32."""
import ctypes as C
import random

import numpy as np
import pytest
import torch

import nabla_amd as nb
from nabla_amd.backend import isa, lib
from nabla_amd.core import engine
from test_rowprog_decode_host import inputs_and_stores, random_program

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_inputs", [6, 8, 9])
@pytest.mark.parametrize("cols", [5, 130, 1003, 4099])
def test_inputs_selected_again_after_a_reduction(hip, n_inputs, cols):
    rng = np.random.default_rng(n_inputs)
    xs = [rng.integers(-9, 10, (33, cols)).astype(np.float32) for _ in range(n_inputs)]

    def f(where, greater, reduce_max, xs):
        v = [greater(xs[k], xs[k - 1]) for k in range(n_inputs)]  # (x0 against the last)
        t = xs[0]
        for k in range(n_inputs):
            t = where(v[k], xs[k], t)
        o = reduce_max(t)
        for k in range(n_inputs):
            o = where(v[k], o, xs[k])
        return o

    engine.clear_plan_cache()
    hip.force_interpreter = True
    try:
        got = f(nb.where, nb.greater, lambda t: nb.reduce_max(t, axis=1, keepdims=True),
                [nb.Tensor.constant(x) for x in xs]).to_torch().cpu()
    finally:
        hip.force_interpreter = False
        engine.clear_plan_cache()
    want = f(torch.where, torch.gt, lambda t: t.max(1, keepdim=True).values, [torch.tensor(x) for x in xs])
    assert torch.equal(got, want)


def run_on_host(rp, mem, rows, cols):
    """The program on float64 arrays [rows, cols], one chunk as long as the row; the largest magnitude."""
    big = 0.0
    reg, acc = {}, {}
    binary = {"add": np.add, "sub": np.subtract, "mul": np.multiply, "gt": np.greater}
    unary = {"neg": np.negative, "relu": lambda a: np.maximum(a, 0.0), "abs": np.abs}
    names = {v: k for k, v in isa.EW.items()}
    fold = [np.sum, np.max, np.min]
    start = [0.0, -np.inf, np.inf]
    row = np.arange(rows, dtype=np.float64)[:, None]
    for i in range(rp.n_ins):
        n = rp.ins[i]
        if n.op == isa.HALT:
            break
        if n.op == isa.BODY:
            continue
        if n.op == isa.ACCINIT:
            acc[n.dst] = np.full((rows, 1), start[n.a])
            continue
        if n.op == isa.ACC:
            part = fold[n.b](np.broadcast_to(reg[n.a], (rows, cols)), axis=1, keepdims=True)
            acc[n.dst] = fold[n.b](np.concatenate([acc[n.dst], part], axis=1), axis=1, keepdims=True)
            continue
        if n.op in (isa.STG, isa.STR):
            if n.op == isa.STG:
                mem[n.dst][:] = reg[n.a]
            else:
                mem[n.dst][:, :1] = reg[n.a]
            continue
        if n.op == isa.LDG:
            v = mem[n.a].copy()
        elif n.op == isa.LDR:
            v = mem[n.a][:, :1].copy()
        elif n.op == isa.IMM:
            v = np.full((rows, 1), rp.imm[n.a])
        elif n.op == isa.COLIDX:
            v = np.arange(cols, dtype=np.float64)[None, :]
        elif n.op == isa.LEADIDX:
            v = row
        elif n.op == isa.RED:
            v = acc[n.a]
        else:
            op = names[n.op]
            a, b, c = (reg.get(r) for r in (n.a, n.b, n.c))
            v = unary[op](a) if op in unary else np.where(a != 0, b, c) if op == "where" else \
                a * b + c if op == "fma" else binary[op](a, b).astype(np.float64)
        reg[n.dst] = np.broadcast_to(v, (rows, v.shape[1])) if v.ndim == 2 else v
        finite = np.abs(v[np.isfinite(v)])
        big = max(big, finite.max() if finite.size else 0.0)
        if not np.isfinite(v).all():
            big = np.inf
    return big


@pytest.mark.parametrize("seed", range(12))
def test_random_programs(hip, seed):
    """Programs of whole numbers through the C interface, in every form that the length of a row
    selects; those whose values leave the whole numbers of float32 are passed over."""
    rng = random.Random(100 + seed)
    ran = 0
    for _ in range(60):
        rp = random_program(rng, exact=True)
        rows, cols = rp.lead_dim[0], rp.C
        gen = np.random.default_rng(rng.randrange(1 << 30))
        loads, stores = inputs_and_stores(rp)
        host = [gen.integers(-3, 4, (rows, cols) if rp.operand[i].lead_stride[0] else (1, cols)).astype(np.float64)
                for i in range(rp.n_operands)]
        # (an operand without a stride between rows is one row that all of them would write)
        if any(host[i].shape[0] == 1 for i in stores) or loads & stores:
            continue
        dev = [torch.tensor(h, dtype=torch.float32).cuda() for h in host]
        want = [np.broadcast_to(h, (rows, cols)).copy() for h in host]
        if run_on_host(rp, want, rows, cols) >= 2.0 ** 24:
            continue
        for i, t in enumerate(dev):
            rp.operand[i].ptr = t.data_ptr()
        rp.reserved = 1  # (the interpreter)
        lib.check(lib.load().nbk_rowprog_launch(C.byref(rp), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        for i in stores:
            np.testing.assert_array_equal(dev[i].cpu().numpy().astype(np.float64), want[i], err_msg=f"operand {i}")
        ran += 1
    assert ran >= 10
