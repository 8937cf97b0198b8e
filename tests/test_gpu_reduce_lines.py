"""Reductions of numbers that lie behind each other (one column), by 16 bytes a lane and by element: around the line
between them, remainders of a workgroup's trip, alone and in a batch.  Sums of whole numbers: exact in float32."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 512), (3, 520), (1, 511), (2, 516), (1, 2048), (1, 8184), (5, 8192), (1, 8190), (1, 16384), (1, 16392), (1, 65536), (300, 1000)]


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("outer,red", SHAPES)
def test_one_column(hip, outer, red, dtype, kind, shift):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(outer + red + kind)
    x = rng.integers(-100, 101, (outer, red)).astype(np.float32)
    buf = torch.full((outer * red + shift + 8,), 1e6, dtype=getattr(torch, dtype), device="cuda")
    buf[shift:shift + outer * red] = torch.tensor(x.reshape(-1)).cuda()
    out = torch.full((outer + 1,), 7.0, device="cuda")
    L, stream = lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    at = buf.data_ptr() + shift * buf.element_size()
    want = [x.sum(1, dtype=np.float64), x.max(1), x.min(1)][kind]
    dt = 1 if dtype == "bfloat16" else 0
    lib.check(L.nbk_reduce_mid(C.c_void_p(at), C.c_void_p(out.data_ptr()), dt, 0, outer, red, 1, kind, stream))
    np.testing.assert_array_equal(out[:-1].cpu().numpy(), want)
    assert out[-1] == 7
    both = torch.zeros((2, outer), device="cuda")
    tasks = (lib.ReduceTask * 2)()
    for t, o in zip(tasks, both):
        t.in_, t.out, t.dtype_in, t.dtype_out, t.outer, t.red, t.inner, t.kind = at, o.data_ptr(), dt, 0, outer, red, 1, kind
    lib.check(L.nbk_reduce_mid_batch(tasks, 2, stream))
    assert torch.equal(both[0], out[:-1]) and torch.equal(both[1], out[:-1])
