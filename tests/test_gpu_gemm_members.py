"""Several products of one left operand in one launch (nbk_gemm_members), on every kernel that carries them: tiles of 64, 128
and 256 in bf16, the guarded one, small and large float32 tiles; with and without biases.  Whole numbers: exact
in float32, and in bf16 as far as they are below 256."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(200, 72, 64), (129, 64, 129), (384, 256, 640), (513, 1000, 96), (2048, 1536, 128)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layout", ["nn", "nt"])
@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("n", [2, 3, 4])
def test_against_the_products_alone(hip, M, N, K, n, layout, dtype):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(M + N + K + n)
    t = getattr(torch, dtype)
    a = torch.tensor(rng.integers(-1, 2, (M, K)) * (rng.random((M, K)) < 0.3), dtype=t).cuda()
    bs = [torch.tensor(rng.integers(-1, 2, (K, N)), dtype=t) for _ in range(n)]
    bias = [torch.tensor(rng.integers(-9, 10, N), dtype=t).cuda() if i % 2 else None for i in range(n)]
    dev = [(b.t().contiguous() if layout == "nt" else b).cuda() for b in bs]
    room = torch.full((n, M * N + 64), 7.0, dtype=t, device="cuda")  # (results in no order of their addresses)
    order = rng.permutation(n)
    d = lib.GemmDesc()
    d.A, d.M, d.N, d.K, d.a_rs, d.a_cs, d.ldc = a.data_ptr(), M, N, K, K, 1, N
    d.b_rs, d.b_cs = (1, K) if layout == "nt" else (N, 1)
    d.batch, d.dtype_ab, d.dtype_c, d.alpha = 1, int(dtype == "bfloat16"), int(dtype == "bfloat16"), 1.0
    p = lib.GemmMembers()
    for i in range(n):
        setattr(p, f"B{i}", dev[i].data_ptr())
        setattr(p, f"bias{i}", None if bias[i] is None else bias[i].data_ptr())
        setattr(p, f"C{i}", room[order[i]].data_ptr())
    L = lib.load()
    at = [C.byref(p, getattr(lib.GemmMembers, f).offset) for f in ("B0", "bias0", "C0")]
    lib.check(L.nbk_gemm_members(C.byref(d), n, *at, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    for i in range(n):
        want = a.double() @ bs[i].double().cuda()
        want = want + bias[i].double() if bias[i] is not None else want
        assert want.abs().max() < 256
        got = room[order[i]]
        assert torch.equal(got[:M * N].view(M, N).double(), want) and (got[M * N:] == 7).all(), i
    d.batch = 2
    assert L.nbk_gemm_members(C.byref(d), n, *at, None) != 0
    d.batch = 1
    assert L.nbk_gemm_members(C.byref(d), 5, *at, None) != 0 and L.nbk_gemm_members(C.byref(d), 1, *at, None) != 0


def launched(lib, a, bs, layout="nn", **fields):
    """Products of ``a`` with each of ``bs`` in one launch (one: nbk_gemm)."""
    M, K = a.shape
    N = bs[0].shape[0] if layout == "nt" else bs[0].shape[1]
    out = torch.full((len(bs), M, N), float("nan"), dtype=a.dtype, device="cuda")
    d = lib.GemmDesc()
    d.A, d.M, d.N, d.K, d.a_rs, d.a_cs, d.ldc = a.data_ptr(), M, N, K, K, 1, N
    d.b_rs, d.b_cs = (1, K) if layout == "nt" else (N, 1)
    code = int(a.dtype == torch.bfloat16)
    d.batch, d.dtype_ab, d.dtype_c, d.alpha = 1, code, code, 1.0
    for field, value in fields.items():
        setattr(d, field, value)
    L, stream = lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if len(bs) == 1:
        d.B, d.C = bs[0].data_ptr(), out.data_ptr()
        lib.check(L.nbk_gemm(C.byref(d), stream))
        return out
    p = lib.GemmMembers()
    for i, b in enumerate(bs):
        setattr(p, f"B{i}", b.data_ptr())
        setattr(p, f"C{i}", out[i].data_ptr())
    at = [C.byref(p, getattr(lib.GemmMembers, f).offset) for f in ("B0", "bias0", "C0")]
    lib.check(L.nbk_gemm_members(C.byref(d), len(bs), *at, stream))
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_batch_strides_are_not_looked_at(hip, dtype):
    """There is no batch: strides left in the description reach neither A nor the choice of a kernel."""
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(1)
    t = getattr(torch, dtype)
    room = torch.randn(4 * 200 * 64, generator=gen, device="cuda").to(t)  # (as far as three strides of A reach)
    a, bs = room[:200 * 64].view(200, 64), [torch.randn(64, 72, generator=gen, device="cuda").to(t) for _ in range(3)]
    got = launched(lib, a, bs, a_bs=200 * 64, b_bs=3, c_bs=5)
    assert torch.equal(got, launched(lib, a, bs)) and not got.isnan().any()


@pytest.mark.parametrize("M,N,K", [(1024, 512, 512), (200, 72, 300), (300, 320, 2100), (500, 400, 131), (513, 1000, 96)])
def test_float32_sums_are_those_of_the_products_alone(hip, M, N, K):
    """Bit for bit, on both sides of the lines between the kernels."""
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(K)
    a, bs = torch.rand(M, K, generator=gen, device="cuda"), [torch.rand(K, N, generator=gen, device="cuda") for _ in range(3)]
    assert torch.equal(launched(lib, a, bs), torch.cat([launched(lib, a, [b]) for b in bs]))


@pytest.mark.parametrize("layout", ["nn", "nt"])
@pytest.mark.parametrize("M,N,K", [(1024, 512, 300), (2048, 1536, 128), (200, 72, 64)])
def test_numbers_without_parts(hip, M, N, K, layout):
    """Infinities and NaN as in the products alone: the second pass of a tile reads the operand of its own product."""
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(N)
    a, bs = torch.randn(M, K, generator=gen, device="cuda"), [torch.randn(K, N, generator=gen, device="cuda") for _ in range(3)]
    a[5, 7] = float("inf")
    bs[1][3, 9], bs[2][K - 1, N - 1] = float("nan"), -3e38
    if layout == "nt":
        bs = [b.t().contiguous() for b in bs]
    got, alone = launched(lib, a, bs, layout), torch.cat([launched(lib, a, [b], layout) for b in bs])
    assert got[1].isnan().any() and got[0].isinf().any()
    assert torch.equal(got.nan_to_num(7e37, 8e37, 9e37), alone.nan_to_num(7e37, 8e37, 9e37))


@pytest.mark.parametrize("K", [8, 40, 56])
def test_bf16_contractions_below_a_tile(hip, K):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(K)
    a, *bs = (torch.tensor(rng.integers(-2, 3, s), dtype=torch.bfloat16).cuda() for s in [(384, K)] + [(K, 256)] * 3)
    for layout in ("nn", "nt"):
        got = launched(lib, a, bs if layout == "nn" else [b.t().contiguous() for b in bs], layout)
        for g, b in zip(got, bs):
            assert torch.equal(g.double(), a.double() @ b.double())
