"""Products x^T dy that share a launch (nbk_gemm_group), in every tile form that their sizes choose, with column sums,
with slices of K of which the last is shorter, and with products that cannot share one.  Whole numbers: every
sum is exact in float32."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K, slices of K)
BF16 = {"64, two buffers": [(64, 8, 96, 1), (200, 72, 500, 1), (8, 120, 333, 1)],
        "64, four buffers": [(4096, 8, 1000, 1), (8, 1024, 1000, 1), (1024, 16, 1000, 2), (8, 4096, 1000, 1)],
        "64 x 128": [(512, 512, 700, 2), (1024, 512, 640, 1), (136, 520, 1000, 1)],
        "128, four buffers": [(512, 1024, 300, 2), (1024, 1024, 200, 1), (264, 520, 130, 1)],
        "128, two buffers": [(1024, 1024, 260, 2), (1024, 2048, 200, 1), (2048, 1032, 130, 1)],
        "eight": [(64 + 8 * i, 72, 100 + i, 1) for i in range(8)]}
F32 = {"16": [(4, 32, 200, 1), (33, 1, 57, 1), (200, 100, 300, 1)],
       "32, eight waves": [(513, 241, 256, 1), (300, 129, 131, 1)],
       "32, four waves": [(500, 400, 131, 1), (400, 600, 100, 1)],
       "out of parts": [(512, 2048, 256, 1), (512, 512, 70, 1), (77, 1000, 33, 1)]}


def run(hip, dtype, problems, colsum=(), plain=None):
    from nabla_amd.backend import lib
    L, stream = lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    rng = np.random.default_rng(sum(map(sum, problems)))
    t = torch.bfloat16 if dtype else torch.float32
    keep, ptrs, want = [], (C.POINTER(lib.GemmDesc) * len(problems))(), []
    for i, (M, N, K, ks) in enumerate(problems):
        a, b = (torch.tensor(rng.integers(-3, 4, s), dtype=t).cuda() for s in ((K, M), (K, N)))
        kc = -(-K // (64 * ks)) * 64 if ks > 1 else K
        out = torch.full((ks, M, N), float("nan"), device="cuda")
        cs = torch.full((ks, N), float("nan"), device="cuda")
        d = lib.GemmDesc()
        d.A, d.B, d.C = a.data_ptr(), b.data_ptr(), out.data_ptr()
        d.M, d.N, d.K, d.a_rs, d.a_cs, d.b_rs, d.b_cs, d.ldc = M, N, kc, 1, M, N, 1, N
        d.batch, d.batch_inner, d.a_bs, d.b_bs, d.c_bs = ks, 1, kc * M, kc * N, M * N
        d.k_last = K - (ks - 1) * kc if ks > 1 else 0
        d.dtype_ab, d.dtype_c, d.alpha = dtype, 0, 1.0
        if i in colsum:
            d.colsum = cs.data_ptr()
        if plain == i:
            d.act = 1
        ptrs[i] = C.pointer(d)
        keep.append((a, b, out, cs, d))
        parts = [(a[k:k + kc].double().t().contiguous() @ b[k:k + kc].double(), b[k:k + kc].double().sum(0)) for k in range(0, K, kc)]
        want.append(parts)
    lib.check(L.nbk_gemm_group(ptrs, len(problems), stream))
    for i, ((a, b, out, cs, d), parts) in enumerate(zip(keep, want)):
        for k, (p, s) in enumerate(parts):
            assert torch.equal(out[k].double(), p.clamp(min=0) if plain == i else p), (i, k)
            assert torch.equal(cs[k].double(), s) if i in colsum else cs[k].isnan().all(), (i, k)


@pytest.mark.parametrize("name", list(BF16))
def test_bf16(hip, name):
    run(hip, 1, BF16[name])
    run(hip, 1, BF16[name], colsum=(0, len(BF16[name]) - 1))


@pytest.mark.parametrize("name", list(F32))
def test_float32(hip, name):
    run(hip, 0, F32[name])


@pytest.mark.parametrize("dtype", [0, 1])
def test_one_that_cannot_share(hip, dtype):
    run(hip, dtype, [(64, 72, 96, 1), (128, 64, 130, 1), (72, 80, 100, 1)], plain=1)
    run(hip, dtype, [(64, 72, 96, 1)])
    if dtype:  # (rows of no whole 16 bytes)
        run(hip, dtype, [(64, 72, 96, 1), (67, 72, 96, 1)])


def test_a_step_reads_its_groups(hip):
    """Weight gradients of a network in one launch, replayed: losses and gradients as from separate steps."""
    import nabla_amd as nb
    from nabla_amd.core import engine
    rng = np.random.default_rng(0)
    sizes = [40, 64, 32, 16, 5]
    ws = [nb.Tensor.constant(rng.standard_normal((a, b)).astype(np.float32) / a ** 0.5) for a, b in zip(sizes, sizes[1:])]

    @nb.compile
    def step(ws, x):
        def loss(ws, x):
            for w in ws:
                x = nb.relu(x @ w)
            return nb.reduce_sum(x * x)
        return nb.value_and_grad(loss)(ws, x)

    for seed in range(4):
        x = np.random.default_rng(seed).standard_normal((90, 40)).astype(np.float32)
        loss, grads = step(ws, nb.Tensor.constant(x))
        tw = [torch.tensor(w.numpy(), dtype=torch.float64, requires_grad=True) for w in ws]
        h = torch.tensor(x, dtype=torch.float64)
        for w in tw:
            h = torch.relu(h @ w)
        (h * h).sum().backward()
        for g, w in zip(grads, tw):
            # (sums of 90 products of three rounded factors: 90 roundings of 2^-24 and a few more)
            assert np.abs(g.numpy() - w.grad.numpy()).max() <= 1e-5 * w.grad.abs().max()
    groups = [s.attrs["group"] for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps if s.attrs.get("group")]
    assert len(groups) >= 4


def products(lib, dtype, pairs, alpha=1.0, together=True):
    """x^T dy of every pair, in one call or one by one."""
    L, stream = lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    outs, ptrs = [], (C.POINTER(lib.GemmDesc) * len(pairs))()
    for i, (a, b) in enumerate(pairs):
        (K, M), N = a.shape, b.shape[1]
        outs.append(torch.full((M, N), float("nan"), device="cuda"))
        d = lib.GemmDesc()
        d.A, d.B, d.C = a.data_ptr(), b.data_ptr(), outs[i].data_ptr()
        d.M, d.N, d.K, d.a_rs, d.a_cs, d.b_rs, d.b_cs, d.ldc = M, N, K, 1, M, N, 1, N
        d.batch, d.batch_inner, d.dtype_ab, d.dtype_c, d.alpha = 1, 1, dtype, 0, alpha
        ptrs[i] = C.pointer(d)
        if not together:
            lib.check(L.nbk_gemm(ptrs[i], stream))
    if together:
        lib.check(L.nbk_gemm_group(ptrs, len(pairs), stream))
    return outs


FORMS = [(512, 512, 1024), (512, 2048, 1024), (200, 100, 300), (64, 64, 3000), (500, 400, 131), (512, 512, 640), (33, 1, 57),
         (128, 32, 2200), (2048, 512, 1024), (400, 600, 100)]


def test_float32_sums_are_those_of_the_products_alone(hip):
    """Bit for bit, whatever else is in the launch."""
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(2)
    pairs = [tuple(torch.rand(K, n, generator=gen, device="cuda") for n in (M, N)) for M, N, K in FORMS]
    for got, alone in zip(products(lib, 0, pairs), products(lib, 0, pairs, together=False)):
        assert torch.equal(got, alone), tuple(got.shape)


@pytest.mark.parametrize("dtype", [0, 1])
def test_scaled(hip, dtype):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(dtype)
    pairs = [tuple(torch.tensor(rng.integers(-3, 4, (K, n)), dtype=torch.bfloat16 if dtype else torch.float32).cuda() for n in (M, N))
             for M, N, K in [(64, 72, 96), (512, 2048, 256), (72, 80, 100), (512, 1024, 33), (400, 600, 100)]]
    for (a, b), got in zip(pairs, products(lib, dtype, pairs, alpha=0.25)):
        assert torch.equal(got.double(), 0.25 * (a.double().t().contiguous() @ b.double()))


def test_bf16_contractions_below_a_tile(hip):
    run(hip, 1, [(64, 72, 40, 1), (128, 64, 8, 1), (72, 80, 56, 1), (512, 520, 24, 1)], colsum=(1, 3))


def test_numbers_without_parts(hip):
    """Infinities and NaN as in the products alone, in every form."""
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(4)
    pairs = [tuple(torch.randn(K, n, generator=gen, device="cuda") for n in (M, N)) for M, N, K in FORMS]
    for i, (a, b) in enumerate(pairs):
        a[i % a.shape[0], i % a.shape[1]] = float("inf")
        b[-1, i % b.shape[1]] = float("nan") if i % 2 else -3e38
    for got, alone in zip(products(lib, 0, pairs), products(lib, 0, pairs, together=False)):
        assert got.isnan().any() or got.isinf().any()
        assert torch.equal(got.nan_to_num(7e37, 8e37, 9e37), alone.nan_to_num(7e37, 8e37, 9e37))
