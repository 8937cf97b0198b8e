"""Every compiled row kernel at sizes, alignments and immediates it was not generated from, against the
interpreter on the same inputs: rows shorter and longer than a lane's chunks, odd ones, operands that
start at an odd element, up to four leading dimensions."""
import ctypes as C

import numpy as np
import pytest
import torch

from nabla_amd.backend import isa, lib, specialize
from test_abi import _program_record

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def programs():
    return [a for _, _, a, _ in specialize.kernels_of(specialize.collect_programs())]


@pytest.mark.parametrize("cols", [1, 2, 3, 4, 7, 100, 255, 333, 1003, 1024, 2052, 4099, 20005])
def test_against_the_interpreter(hip, programs, cols):
    rng = np.random.default_rng(cols)
    L = lib.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    compared = 0
    for a in programs:
        if a["n_stage"] and cols > 4096:
            a = dict(a, n_stage=0, operands=[type(o)(**{**vars(o), "stage_slot": -1}) for o in a["operands"]])
        rp = _program_record(a)
        dims = [3, 2, 5, 2][:rp.n_lead]
        rows = int(np.prod(dims)) if dims else 1
        rp.C, rp.block = cols, 64 if cols <= 1024 else 256 if cols <= 4096 else 512
        for k, d in enumerate(dims):
            rp.lead_dim[k] = d
        for i in range(rp.n_imm):
            if rp.imm[i] > 1.5:  # (the length that a mean divides by; small ones are epsilons and flags)
                rp.imm[i] = float(cols + 1)
        keep, outs = [], []
        written = {i[1] for i in a["ins"] if i[0] in (isa.STG, isa.STR)}
        for i, o in enumerate(a["operands"]):
            od = rp.operand[i]
            od.vec_ok = 0
            at, strides = (cols if o.col_stride else 1), []
            for d, s in reversed(list(zip(dims, o.lead_strides))):
                strides.insert(0, at if s else 0)
                at *= d if s else 1
            for k, s in enumerate(strides):
                od.lead_stride[k] = s
            n, dt = max(at, 1), o.dtype.to_torch()
            if o.dtype.is_float():
                x = torch.tensor(rng.standard_normal(n + 1)).to(dt)
            else:
                x = torch.tensor(rng.integers(0, 2 if dt in (torch.bool, torch.uint8) else cols + 1, n + 1)).to(dt)
            x = x.cuda()
            keep.append(x)
            od.ptr = x.data_ptr() + x.element_size()  # (an odd element)
            if i in written:
                outs.append((i, x))
        results = []
        for reserved in (0, 1):
            for i, x in outs:
                x.zero_()
            rp.reserved = reserved
            if not reserved:
                assert L.nbk_rowprog_is_specialized(C.byref(rp)) >= 1
            lib.check(L.nbk_rowprog_launch(C.byref(rp), st))
            results.append([x.clone() for _, x in outs])
        for (i, x), got, want in zip(outs, *results):
            name = f"{specialize.program_hash(a):016x} operand {i} ({' '.join(a['members'])[:60]})"
            if not x.dtype.is_floating_point:
                assert torch.equal(got, want), name
                continue
            g, w = got.double(), want.double()
            same = (g == w) | (g.isnan() & w.isnan())
            # two roundings of a bf16 result, or the hardware functions that programs of bf16 results use
            # (1e-4); float32: sums in another order, up to 2e-5 of the largest value behind a cancellation
            tol = (2.0 ** -7 if x.dtype == torch.bfloat16 else 2e-4 if any(
                o.dtype.to_torch() == torch.bfloat16 for o in a["operands"]) else 2e-5)
            scale = torch.where(w.isfinite(), w.abs(), 0).max()
            assert (same | ((g - w).abs() <= tol * torch.maximum(w.abs(), scale))).all(), name
            compared += 1
        assert rows >= 1
    assert compared >= 30


def test_functions_are_the_interpreters(hip, programs):
    """Programs without reductions at an alignment that no benchmark step has: bit for bit."""
    L = lib.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    rng = np.random.default_rng(0)
    n, compared = 4099, 0
    for a in programs:
        rp = _program_record(a)
        if rp.has_reduce or any(o.col_stride == 0 or not o.dtype.is_float() for o in a["operands"]):
            continue
        rp.n_lead, rp.C = 1, n
        rp.lead_dim[0] = 1
        written = {i[1] for i in a["ins"] if i[0] in (isa.STG, isa.STR)}
        keep, outs = [], []
        for i, o in enumerate(a["operands"]):
            x = (torch.tensor(rng.standard_normal(n + 1)) * 3).to(o.dtype.to_torch()).cuda()
            keep.append(x)
            od = rp.operand[i]
            od.vec_ok, od.ptr, od.col_stride = 0, x.data_ptr() + x.element_size(), 1
            for k in range(4):
                od.lead_stride[k] = 0
            if i in written:
                outs.append(x)
        results = []
        for rp.reserved in (0, 1):
            for x in outs:
                x.zero_()
            assert rp.reserved or L.nbk_rowprog_is_specialized(C.byref(rp)) == 1
            lib.check(L.nbk_rowprog_launch(C.byref(rp), st))
            results.append([x.clone() for x in outs])
        for got, want in zip(*results):
            same = (got == want) | (got.isnan() & want.isnan())
            assert same.all(), f"{specialize.program_hash(a):016x} ({' '.join(a['members'])[:60]})"
        compared += 1
    assert compared >= 40
