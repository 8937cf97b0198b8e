"""bf16 products at the sizes where the 64 x 64 tile, the left-over of a contraction that is no
multiple of 64, unequal slices of it and rows at odd elements can go wrong."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    from nabla_amd.backend import lib
    return lib.load()


def product(L, M, N, K, layout, ks=1, colsum=False, odd=0):
    """A product of random integers (their sums are exact in float32) and its column sums of B."""
    from nabla_amd.backend import lib
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = rng.integers(-4, 5, (M, K)).astype(np.float32), rng.integers(-4, 5, (K, N)).astype(np.float32)

    def put(x, transposed):
        x = np.ascontiguousarray(x.T if transposed else x)
        buf = torch.zeros(x.shape[0], x.shape[1] + odd, dtype=torch.bfloat16)
        buf[:, :x.shape[1]] = torch.tensor(x)
        return buf.cuda(), x.shape[1] + odd

    ad, lda = put(a, layout[0] == "t")
    bd, ldb = put(b, layout[1] == "t")
    d = lib.GemmDesc()
    kc = -(-K // (64 * ks)) * 64 if ks > 1 else K
    out = torch.full((ks, M, N), float("nan"), device="cuda")
    cs = torch.full((ks, N), float("nan"), device="cuda")
    d.A, d.B, d.C = ad.data_ptr(), bd.data_ptr(), out.data_ptr()
    d.M, d.N, d.K = M, N, kc
    d.k_last = K - (ks - 1) * kc if ks > 1 else 0
    d.a_rs, d.a_cs = (1, lda) if layout[0] == "t" else (lda, 1)
    d.b_rs, d.b_cs = (1, ldb) if layout[1] == "t" else (ldb, 1)
    d.ldc, d.batch, d.batch_inner = N, ks, 1
    d.a_bs, d.b_bs, d.c_bs = kc * d.a_cs, kc * d.b_rs, M * N
    d.dtype_ab, d.dtype_c, d.alpha = 1, 0, 1.0
    if colsum:
        d.colsum = cs.data_ptr()
    lib.check(L.nbk_gemm(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    np.testing.assert_array_equal(out.sum(0).cpu().numpy(), a @ b)
    if colsum:
        np.testing.assert_array_equal(cs.sum(0).cpu().numpy(), b.sum(0))


@pytest.mark.parametrize("M,N,K", [(8, 8, 1), (64, 64, 63), (72, 136, 65), (200, 64, 127), (512, 1024, 333), (1600, 1600, 70)])
@pytest.mark.parametrize("colsum", [False, True])
def test_left_over_of_the_contraction(L, M, N, K, colsum):
    product(L, M, N, K, "tn", colsum=colsum)


@pytest.mark.parametrize("K,ks", [(4100, 4), (1030, 2), (257, 2), (129, 3)])
@pytest.mark.parametrize("M,N", [(72, 200), (1032, 1048)])
def test_unequal_slices(L, M, N, K, ks):
    product(L, M, N, K, "tn", ks=ks, colsum=True)
    product(L, M + 1, N + 3, K, "nt", ks=ks)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(8, 8, 64), (56, 72, 128), (128, 64, 192), (333, 520, 256)])
def test_small_tiles(L, layout, M, N, K):
    product(L, M - M % 8, N, K, layout)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("odd", [1, 2, 4])
def test_rows_at_odd_elements(L, layout, odd):
    product(L, 131, 77, 83, layout, odd=odd)
