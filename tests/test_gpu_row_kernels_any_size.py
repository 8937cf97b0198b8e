"""Every compiled row kernel, in every form that it has, at sizes, alignments and immediates it was not
generated from, against the interpreter on the same inputs: rows shorter and longer than a lane's chunks, odd
ones, operands that start at an odd element, up to four leading dimensions."""
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
        if a["n_stage"] and cols > 4096:  # (longer than what the generic form stages: in test_every_form)
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
    assert compared >= 30


def form(a, generic, rp):
    """What nbk_rowprog_launch runs of a kernel for a reduction program (the rule in rowprog.hip)."""
    chunks = -(-rp.C // 4)
    need = -(-chunks // rp.block)
    cpt = next((c for c in (1, 2, 4, 8) if need <= c), 0)
    if cpt in specialize.resident_variants(a):
        if rp.C != 4 * cpt * rp.block:
            return cpt, "masked"
        rows = int(np.prod([rp.lead_dim[k] for k in range(rp.n_lead)]))
        moved = sum(rows * rp.C * o.dtype.size_in_bytes for o in generic["operands"] if o.col_stride)
        return cpt, "stream" if moved > 256 << 20 else "full"
    if specialize.stage16_operand(generic) is not None and rp.n_stage == 0 and rp.C % 4 == 0:
        return 0, "stage16"
    return 0, "generic"


def streams(generic):
    """Whether rows enough for the streaming forms can be had."""
    return bool(generic["lead"]) and any(o.col_stride for o in generic["operands"])


def launches(a, generic):
    """(row length, workgroup, whether to exceed the last-level cache) for every form of the kernel."""
    cpts = specialize.resident_variants(a)
    for cpt in cpts:
        yield 4 * cpt * 64 - 8, 64, False
        yield 4 * cpt * 64, 64, False
        if streams(generic):
            yield 4 * cpt * 256, 256, True
    yield 4 * cpts[-1] * 64 + (8 if "approx_hash" in a else 5), 64, False  # (the generic form)
    if specialize.stage16_operand(generic) is not None:
        yield 4 * cpts[-1] * 64 + 8, 64, False


def test_every_form(hip):
    L = lib.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    gen = torch.Generator(device="cuda").manual_seed(0)
    pool = torch.randn(80 << 20, generator=gen, device="cuda")
    kernels = [k for k in specialize.kernels_of(specialize.collect_programs()) if k[2]["has_reduce"]]
    assert len(kernels) >= 60
    for _, name, a, generic in kernels:
        ran = set()
        # the kernels of one program alone are found by its alignment, too; the others start at an odd element
        shift = 0 if "approx_hash" in a else 1
        for cols, block, large in launches(a, generic):
            rp = _program_record(generic)
            rp.C, rp.block = cols, block
            dims = [1] * rp.n_lead
            if dims:
                dims[0], dims[-1] = 2, dims[-1] * 5
            if large:
                per_row = sum(cols * o.dtype.size_in_bytes for o in generic["operands"] if o.col_stride)
                dims[-1] = (256 << 20) // (per_row * int(np.prod(dims[:-1]))) + 3
            for k, d in enumerate(dims):
                rp.lead_dim[k] = d
            written = {i[1] for i in a["ins"] if i[0] in (isa.STG, isa.STR)}
            operands, outs = [], []
            for i, o in enumerate(generic["operands"]):
                od = rp.operand[i]
                at, strides = (cols if o.col_stride else 1), []
                for d, s in reversed(list(zip(dims, o.lead_strides))):
                    strides.insert(0, at if s else 0)
                    at *= d if s else 1
                for k, s in enumerate(strides):
                    od.lead_stride[k] = s
                dt = o.dtype.to_torch()
                if o.dtype.is_float():
                    n = at + shift
                    x = torch.cat([pool] * -(-n // pool.numel()))[:n].to(dt) if n > pool.numel() else pool[i * 3:n + i * 3].to(dt)
                    if x.data_ptr() % 16 or x._base is not None or i in written:
                        x = x.clone()
                else:
                    x = torch.randint(0, 2 if dt in (torch.bool, torch.uint8) else cols + 1, (at + shift,), generator=gen, device="cuda").to(dt)
                operands.append(x)
                od.ptr = x.data_ptr() + shift * x.element_size()
                od.vec_ok = 0 if shift else int(o.vec_ok)
                if i in written:
                    outs.append(x)
            results = []
            for rp.reserved in (0, 1):
                for x in outs:
                    x.zero_()
                assert rp.reserved or L.nbk_rowprog_is_specialized(C.byref(rp)) == (3 if "approx_hash" in a else 1), name
                lib.check(L.nbk_rowprog_launch(C.byref(rp), st))
                results.append([x.clone() for x in outs])
            what = form(a, generic, rp)
            ran.add(what)
            for got, want in zip(*results):
                where = f"{name} {what} C {cols} ({' '.join(a['members'])[:60]})"
                if not got.dtype.is_floating_point:
                    assert torch.equal(got, want), where
                    continue
                # (tolerances as above)
                tol = (2.0 ** -7 if got.dtype == torch.bfloat16 else 2e-4 if any(
                    o.dtype.to_torch() == torch.bfloat16 for o in a["operands"]) else 2e-5)
                g, w = got.float(), want.float()
                same = (g == w) | (g.isnan() & w.isnan())
                scale = torch.where(w.isfinite(), w.abs(), 0).max()
                assert (same | ((g - w).abs() <= tol * torch.maximum(w.abs(), scale))).all(), where
        forms = {(c, f) for c in specialize.resident_variants(a) for f in ("masked", "full") + (("stream",) if streams(generic) else ())}
        forms.add((0, "generic"))
        if specialize.stage16_operand(generic) is not None:
            forms.add((0, "stage16"))
        assert ran == forms, name


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
