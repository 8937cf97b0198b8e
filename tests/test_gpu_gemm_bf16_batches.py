"""Batches of bf16 products of at most one 128 x 128 tile each, on both sides of the line between the
tiles.  Whole numbers: every sum is exact in float32."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("batch,M,N,K", [(64, 104, 104, 64), (65, 104, 104, 64), (65, 128, 128, 512), (66, 128, 128, 448),
                                         (300, 64, 64, 64), (130, 72, 64, 128), (140, 64, 120, 192), (70, 128, 72, 576)])
def test_members_of_one_tile(hip, layout, batch, M, N, K):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(M + N + K)
    a, b = (torch.tensor(rng.integers(-4, 5, s).astype(np.float32)) for s in ((batch, M, K), (batch, K, N)))
    ad = (a.transpose(1, 2).contiguous() if layout[0] == "t" else a).to(torch.bfloat16).cuda()
    bd = (b.transpose(1, 2).contiguous() if layout[1] == "t" else b).to(torch.bfloat16).cuda()
    out = torch.full((batch, M, N), float("nan"), device="cuda")
    d = lib.GemmDesc()
    d.A, d.B, d.C = ad.data_ptr(), bd.data_ptr(), out.data_ptr()
    d.M, d.N, d.K = M, N, K
    d.a_rs, d.a_cs = (1, M) if layout[0] == "t" else (K, 1)
    d.b_rs, d.b_cs = (1, K) if layout[1] == "t" else (N, 1)
    d.ldc, d.batch, d.batch_inner, d.a_bs, d.b_bs, d.c_bs = N, batch, 1, M * K, K * N, M * N
    d.dtype_ab, d.dtype_c, d.alpha = 1, 0, 1.0
    lib.check(lib.load().nbk_gemm(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    np.testing.assert_array_equal(out.cpu().numpy(), np.matmul(a.numpy(), b.numpy()))
