"""bf16 products whose K loop runs over four tile buffers: contractions around the number of buffers and
with a left-over tile in front, the three tiles that are pipelined that deep, slices and column sums,
further operand pairs as first and last tiles.  Whole numbers: every sum is exact in float32."""
import ctypes as C

import numpy as np
import pytest
import torch

from test_gpu_gemm_small_tiles import L, product  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(8, 8, 576), (72, 200, 640), (520, 512, 704),     # 64 x 64
                                   (1104, 1048, 512), (1160, 136, 4096), (2000, 520, 576),  # 64 x 128
                                   (1672, 1544, 320), (2048, 2048, 384), (1800, 1600, 448)])  # 128 x 128
def test_layouts(L, layout, M, N, K):  # noqa: F811
    product(L, M, N, K, layout)


@pytest.mark.parametrize("M,N,K", [(72, 136, 577), (520, 512, 1087), (1104, 1048, 513), (1104, 1048, 700),
                                   (1672, 1544, 321), (1600, 1600, 383)])
@pytest.mark.parametrize("colsum", [False, True])
def test_left_over_tile(L, M, N, K, colsum):  # noqa: F811
    product(L, M, N, K, "tn", colsum=colsum)


@pytest.mark.parametrize("M,N,K,ks", [(72, 200, 1800, 3), (520, 512, 4100, 2), (1104, 520, 2500, 3), (1160, 1160, 700, 2)])
def test_slices(L, M, N, K, ks):  # noqa: F811
    product(L, M, N, K, "tn", ks=ks, colsum=True)


@pytest.mark.parametrize("M,N,K", [(128, 128, 576), (1104, 1048, 512), (1672, 1544, 320)])
@pytest.mark.parametrize("bkc", [False, True])
@pytest.mark.parametrize("extra", [[16], [64, 8], [128], [16, 64, 192], [8, 24, 64, 128]])
def test_operand_pairs(L, M, N, K, bkc, extra):  # noqa: F811
    from nabla_amd.backend import lib
    rng = np.random.default_rng(M + K + sum(extra))
    want, keep = 0, []

    def pair(k, rows=0):
        """Operands [M, k] and [k, N] with the strides of the base product where it is a deep pair."""
        a, b = rng.integers(-3, 4, (M, k)).astype(np.float32), rng.integers(-3, 4, (k, N)).astype(np.float32)
        ld = max(rows, k)
        ad = torch.zeros(M, ld, dtype=torch.bfloat16)
        ad[:, :k] = torch.tensor(a)
        if bkc:
            bd = torch.zeros(N, ld, dtype=torch.bfloat16)
            bd[:, :k] = torch.tensor(b.T.copy())
        else:
            bd = torch.tensor(b).to(torch.bfloat16)
        ad, bd = ad.cuda(), bd.cuda()
        keep.append((ad, bd))
        return a @ b, ad, bd, (ld, 1), ((1, ld) if bkc else (N, 1))

    d = lib.GemmDesc()
    p, ad, bd, sa, sb = pair(K)
    want = want + p
    out = torch.full((M, N), float("nan"), device="cuda")
    d.A, d.B, d.C = ad.data_ptr(), bd.data_ptr(), out.data_ptr()
    d.M, d.N, d.K, d.ldc, d.batch, d.batch_inner = M, N, K, N, 1, 1
    (d.a_rs, d.a_cs), (d.b_rs, d.b_cs) = sa, sb
    d.dtype_ab, d.dtype_c, d.alpha, d.n_terms = 1, 0, 1.0, len(extra)
    for i, k in enumerate(extra):
        p, ad, bd, sa, sb = pair(k, K if k > 64 else 0)
        want = want + p
        t = d.term[i]
        t.A, t.B, t.K = ad.data_ptr(), bd.data_ptr(), k
        (t.a_rs, t.a_cs), (t.b_rs, t.b_cs) = sa, sb
    lib.check(L.nbk_gemm(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    np.testing.assert_array_equal(out.cpu().numpy(), want)
