"""Reductions over a middle axis at the edges of their strips: rows shorter and longer than a strip of
every width, row counts around what a workgroup takes abreast and keeps in flight, every element type
and alignment.  Whole numbers below 2^24: float32 sums are exact in any order."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TYPES = {"f32": (0, torch.float32), "bf16": (1, torch.bfloat16), "f16": (2, torch.float16), "u8": (5, torch.uint8)}
SHAPES = [(1, 1, 1), (1, 300, 1), (5, 7, 3), (1, 255, 4), (1, 257, 8), (2, 64, 12), (1, 2049, 33), (3, 31, 40),
          (1, 33, 63), (1, 200, 65), (7, 9, 127), (1, 100, 516), (40, 17, 264), (1, 6, 1032), (300, 3, 257),
          (65537, 2, 4), (1, 9, 65536), (1, 8, 65540), (2, 40, 8200), (1, 1, 5000)]


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("outer,red,inner", SHAPES)
def test_strips(hip, dtype, outer, red, inner):
    from nabla_amd.backend import lib
    L = lib.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    code, tdt = TYPES[dtype]
    rng = np.random.default_rng(red + inner)
    lo = 0 if dtype == "u8" else -100
    x = rng.integers(lo, 101, (outer, red, inner))
    for shift in (0, 1):  # an operand that starts on 16 bytes and one that does not
        buf = torch.full((x.size + shift + 1,), 99, dtype=tdt, device="cuda")
        buf[shift:-1] = torch.tensor(x).to(tdt).reshape(-1).cuda()
        for kind, want in ((0, x.sum(1)), (1, x.max(1)), (2, x.min(1))):
            out = torch.full((outer * inner + 1 + shift,), 7.5, device="cuda")
            lib.check(L.nbk_reduce_mid(C.c_void_p(buf.data_ptr() + shift * buf.element_size()),
                                       C.c_void_p(out.data_ptr() + 4 * shift), code, 0, outer, red, inner, kind, st))
            got = out.cpu().numpy()
            np.testing.assert_array_equal(got[shift:-1].reshape(outer, inner), want.astype(np.float32))
            assert got[-1] == 7.5 and (shift == 0 or got[0] == 7.5)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("outer,red,inner", [(65535 + 100, 24, 33), (65535 + 40, 40, 64), (600, 70, 33)])
def test_one_order_of_additions(hip, dtype, outer, red, inner):
    """Alone or in a launch with others, and past the 65535 members that one launch's grid holds: the same bits, and
    members of the same numbers the same results."""
    from nabla_amd.backend import lib
    L = lib.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    code, tdt = TYPES[dtype]
    one = torch.randn((1, red, inner), generator=torch.Generator().manual_seed(0)).to(tdt).cuda()
    x = one.expand(outer, red, inner).contiguous()
    alone, batched = (torch.empty((outer, inner), device="cuda") for _ in range(2))
    lib.check(L.nbk_reduce_mid(C.c_void_p(x.data_ptr()), C.c_void_p(alone.data_ptr()), code, 0, outer, red, inner, 0, st))
    task = lib.ReduceTask()
    task.in_, task.out = x.data_ptr(), batched.data_ptr()
    task.dtype_in, task.dtype_out, task.kind = code, 0, 0
    task.outer, task.red, task.inner = outer, red, inner
    lib.check(L.nbk_reduce_mid_batch(C.byref(task), 1, st))
    assert torch.equal(alone, batched)
    assert torch.equal(alone, alone[:1].expand(outer, inner))


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("outer,red,inner", [(64, 1024, 4099), (1024, 12, 1000), (8, 1000, 30011), (1030, 130, 1024),
                                             (3, 2000, 20), (1, 4096, 64)])
def test_long_axes_are_not_one_chain(hip, dtype, outer, red, inner):
    """Sums of uniform numbers against float64.  A sum of n equal shares in one chain is rounded once a share, at
    about half of its value on the average: sqrt(n) / 3 of 2^-24 of it.  In sixteen chains, or in two that take
    four numbers at a time, the longest axis here keeps below 2^-23; one chain has 10 * 2^-24."""
    from nabla_amd.backend import lib
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    code, tdt = TYPES[dtype]
    x = torch.rand((outer, red, inner), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").to(tdt)
    out = torch.empty((outer, inner), device="cuda")
    lib.check(lib.load().nbk_reduce_mid(C.c_void_p(x.data_ptr()), C.c_void_p(out.data_ptr()), code, 0, outer, red, inner, 0, st))
    off = size = 0.0
    for got, rows in zip(out, x):
        want = rows.sum(0, dtype=torch.float64)
        off, size = off + ((got - want) ** 2).sum(), size + (want ** 2).sum()
    assert (off / size) ** 0.5 <= 2.0 ** -23
