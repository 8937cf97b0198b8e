"""float32 products out of bf16 parts: every layout at the edges of both tiles and of a K tile of 32, slices,
epilogues, against float64; numbers that have no parts (infinities, NaN, beyond the largest bf16)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def product(a, b, layout, alpha=1.0, **fields):
    from nabla_amd.backend import lib
    M, K = a.shape
    N = b.shape[1]
    ad = torch.tensor(np.ascontiguousarray(a.T if layout[0] == "t" else a)).cuda()
    bd = torch.tensor(np.ascontiguousarray(b.T if layout[1] == "t" else b)).cuda()
    out = torch.full((M, N), float("nan"), device="cuda")
    d = lib.GemmDesc()
    d.A, d.B, d.C = ad.data_ptr(), bd.data_ptr(), out.data_ptr()
    d.M, d.N, d.K = M, N, K
    d.a_rs, d.a_cs = (1, M) if layout[0] == "t" else (K, 1)
    d.b_rs, d.b_cs = (1, K) if layout[1] == "t" else (N, 1)
    d.ldc, d.batch, d.batch_inner, d.dtype_ab, d.dtype_c, d.alpha = N, 1, 1, 0, 0, alpha
    for name, value in fields.items():
        setattr(d, name, value)
    lib.check(lib.load().nbk_gemm(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return out.cpu().numpy()


# A sum is rounded once per K tile of 32 and accumulator (2^-24 of what has been summed, at most the sum of
# magnitudes), the five small products as often at 2^-8 of their size, and three additions at the end; what the six
# products leave out is up to 2^-24 of one.
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(1025, 769, 31), (897, 1024, 64), (1100, 1200, 65), (1024, 1000, 129),   # 64 x 64
                                   (2047, 2050, 95), (2100, 1990, 160), (4097, 1921, 33)])                 # 128 x 128
def test_against_float64(hip, layout, M, N, K):
    rng = np.random.default_rng(K)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (K, N)))
    bias = rng.standard_normal(N).astype(np.float32)
    bd = torch.tensor(bias).cuda()
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want, size = a64 @ b64, np.abs(a64) @ np.abs(b64)
    tol = (-(-K // 32) + 4) * 2.0 ** -24 * size + 2.0 ** -23 * np.abs(want)
    assert (np.abs(product(a, b, layout) - want) <= tol).all()
    got = product(a, b, layout, alpha=0.5, bias=bd.data_ptr(), act=1)  # relu
    want = np.maximum(0.5 * want + bias, 0.0)
    assert (np.abs(got - want) <= tol + 2.0 ** -23 * (np.abs(want) + np.abs(bias))).all()


@pytest.mark.parametrize("M,N", [(1024, 1024), (2048, 2048)])
@pytest.mark.parametrize("x", [1 + 2.0 ** -8 - 2.0 ** -17, 1 - 2.0 ** -8 + 2.0 ** -17, 1 + 2.0 ** -9 + 2.0 ** -18])
def test_numbers_whose_left_out_products_add_up(hip, M, N, x):
    """All of one sign and size: x2 y3 + x3 y2 are 2^-24 of the first product, K times over."""
    K = 96
    a, b = np.full((M, K), x, np.float32), np.full((K, N), x, np.float32)
    want = K * float(np.float32(x)) ** 2
    tol = (-(-K // 32) + 4) * 2.0 ** -24 * want + 2.0 ** -23 * want
    assert (np.abs(product(a, b, "nn") - want) <= tol).all()


@pytest.mark.parametrize("M,N", [(1024, 1024), (2048, 2048)])
@pytest.mark.parametrize("e,f", [(-30, 40), (-112, 60), (-126, 70), (-140, 80), (-145, 100), (40, 50), (100, -100),
                                 (120, -30), (-70, -60)])
def test_numbers_of_every_size(hip, M, N, e, f):
    """Operands about 2^e and 2^f, down to the smallest float32 and up to sums near the largest."""
    K = 70
    rng = np.random.default_rng(K)
    a, b = (np.ldexp(rng.standard_normal(s), x).astype(np.float32) for s, x in (((M, K), e), ((K, N), f)))
    for x, y in ((a, b), (b.T, a.T)):
        x64, y64 = x.astype(np.float64), y.astype(np.float64)
        want, size = x64 @ y64, np.abs(x64) @ np.abs(y64)
        # as above, for numbers whose last digit may be 2^-149 (the sum is one of float32 numbers itself)
        tol = (-(-K // 32) + 4) * 2.0 ** -24 * size + 2.0 ** -23 * np.abs(want) + K * 2.0 ** -149
        assert (np.abs(product(np.ascontiguousarray(x), np.ascontiguousarray(y), "nn") - want) <= tol).all()


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N", [(1024, 1024), (2048, 2048), (1025, 897)])
def test_a_contraction_of_one_number_is_rounded_once(hip, M, N, layout):
    rng = np.random.default_rng(M)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((M, 1), (1, N)))
    np.testing.assert_array_equal(product(a, b, layout), a * b)
    bias = rng.standard_normal(N).astype(np.float32)
    bd = torch.tensor(bias).cuda()
    np.testing.assert_array_equal(product(a, b, layout, bias=bd.data_ptr(), act=1), np.maximum(a * b + bias, 0))


@pytest.mark.parametrize("M,N", [(1024, 1024), (2048, 2048)])
def test_numbers_without_parts(hip, M, N):
    K = 70
    rng = np.random.default_rng(0)
    a, b = (rng.uniform(0.5, 1.0, s).astype(np.float32) for s in ((M, K), (K, N)))
    a[3, 5], a[70, 69], b[11, 20] = np.inf, -np.inf, np.nan
    a[9, 1], b[1, 30] = np.inf, 0.0                     # (infinity times zero)
    a[M - 1, 0], b[0, N - 1] = 3.4e38, 1e-30             # rounds to infinity as a bf16
    a[40, :] = 1e37                                      # a sum beyond the largest float32
    want = np.zeros((M, N), np.float32)
    with np.errstate(all="ignore"):
        for k in range(K):
            want += a[:, k:k + 1] * b[k:k + 1]
    got = product(a, b, "nn")
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= 1e-5 * np.abs(want[ok])).all()


def seconds(f, n=20):
    f()
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    a.record()
    for _ in range(n):
        f()
    b.record()
    b.synchronize()
    return a.elapsed_time(b)


@pytest.mark.parametrize("layout", ["nn", "tn"])
def test_numbers_without_parts_cost_one_more_pass(hip, layout):
    """A product of NaN throughout: every wave runs its tile again on the float32 instruction, which has a
    third of the rate (one result after the other took 46 times as long)."""
    from nabla_amd.backend import lib
    n = 1024
    out = torch.empty((n, n), device="cuda")
    times = []
    for value in (1.0, float("nan")):
        x = torch.full((n, n), value, device="cuda")
        d = lib.GemmDesc()
        d.A, d.B, d.C = x.data_ptr(), x.data_ptr(), out.data_ptr()
        d.M, d.N, d.K = n, n, n
        d.a_rs, d.a_cs = (1, n) if layout[0] == "t" else (n, 1)
        d.b_rs, d.b_cs, d.ldc, d.batch, d.batch_inner, d.alpha = n, 1, n, 1, 1, 1.0
        st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        times.append(seconds(lambda: lib.check(lib.load().nbk_gemm(C.byref(d), st))))
        assert torch.isnan(out).all() == (value != value)
    assert times[1] <= 8 * times[0]
