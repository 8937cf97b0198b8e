"""float32 products whose last tile holds fewer rows or columns than a piece of a load, as many, and
one more, in every layout and tile size.  Whole numbers: every sum is exact in float32.  Whatever stands
behind a row of an operand is NaN: none of it may reach a result."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(m, n, k) for m, n in [(1, 3), (2, 1), (3, 2), (4, 5), (5, 4), (33, 34), (35, 67), (63, 31)] for k in (3, 64, 131)]
SIZES += [(1473, 1475, 35), (1474, 1474, 32), (2817, 2945, 17), (2818, 2947, 16)]  # 64 x 64 tiles
SIZES += [(3969, 1923, 257), (3970, 1922, 256), (3971, 1921, 290), (4096, 2048, 259)]  # 128 x 128 tiles


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_edges(hip, M, N, K, layout):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(M + 3 * N + K)
    a, b = (rng.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (K, N)))

    def put(x, transposed):
        x = torch.tensor(x.T.copy() if transposed else x)
        buf = torch.full((x.shape[0] + 1, x.shape[1] + 3), float("nan"))
        buf[:-1, :-3] = x
        return buf.cuda(), buf.shape[1]

    (ad, lda), (bd, ldb) = put(a, layout[0] == "t"), put(b, layout[1] == "t")
    out = torch.full((M + 1, N + 1), 7.0, device="cuda")
    d = lib.GemmDesc()
    d.A, d.B, d.C = ad.data_ptr(), bd.data_ptr(), out.data_ptr()
    d.M, d.N, d.K = M, N, K
    d.a_rs, d.a_cs = (1, lda) if layout[0] == "t" else (lda, 1)
    d.b_rs, d.b_cs = (1, ldb) if layout[1] == "t" else (ldb, 1)
    d.ldc, d.batch, d.batch_inner, d.dtype_ab, d.dtype_c, d.alpha = N + 1, 1, 1, 0, 0, 1.0
    lib.check(lib.load().nbk_gemm(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:M, :N], a @ b)
    assert (got[M] == 7).all() and (got[:, N] == 7).all()
