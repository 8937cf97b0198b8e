"""float32 products at the sizes where the tiles, the left-over of a K tile, rows at any element, two
batch levels and the epilogue can go wrong.  Random integers: every sum is exact in float32."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    from nabla_amd.backend import lib
    return lib.load()


def product(L, M, N, K, layout, batch=(1, 1), odd=0, epilogue=False):
    from nabla_amd.backend import lib
    nb = batch[0] * batch[1]
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = rng.integers(-4, 5, (nb, M, K)).astype(np.float32), rng.integers(-4, 5, (nb, K, N)).astype(np.float32)

    def put(x, transposed):
        x = np.ascontiguousarray(x.transpose(0, 2, 1) if transposed else x)
        buf = torch.zeros(x.shape[0], x.shape[1], x.shape[2] + odd)
        buf[:, :, :x.shape[2]] = torch.tensor(x)
        return buf.cuda(), x.shape[2] + odd

    ad, lda = put(a, layout[0] == "t")
    bd, ldb = put(b, layout[1] == "t")
    out = torch.full((nb, M, N + 2), float("nan"), device="cuda")
    d = lib.GemmDesc()
    d.A, d.B, d.C = ad.data_ptr(), bd.data_ptr(), out.data_ptr()
    d.M, d.N, d.K = M, N, K
    d.a_rs, d.a_cs = (1, lda) if layout[0] == "t" else (lda, 1)
    d.b_rs, d.b_cs = (1, ldb) if layout[1] == "t" else (ldb, 1)
    d.ldc, d.batch, d.batch_inner = N + 2, nb, batch[1]
    steps = (ad[0].numel(), bd[0].numel(), out[0].numel())
    d.a_bs, d.b_bs, d.c_bs = (s * batch[1] for s in steps)
    d.a_bs2, d.b_bs2, d.c_bs2 = steps
    if batch[1] == 1:
        d.a_bs, d.b_bs, d.c_bs = steps
    d.dtype_ab, d.dtype_c, d.alpha = 0, 0, 1.0
    want = a @ b
    if epilogue:
        bias, res = rng.integers(-9, 10, N).astype(np.float32), rng.integers(-9, 10, out.shape).astype(np.float32)
        bias_d, res_d = torch.tensor(bias).cuda(), torch.tensor(res).cuda()
        d.bias, d.residual, d.alpha, d.act = bias_d.data_ptr(), res_d.data_ptr(), 2.0, 1
        want = np.maximum(2.0 * want + bias, 0.0) + res[:, :, :N]
    lib.check(L.nbk_gemm(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:, :, :N], want)
    assert np.isnan(got[:, :, N:]).all()


SIZES = [(1, 1, 1), (32, 32, 64), (33, 31, 65), (200, 32, 3), (129, 65, 784), (513, 700, 63), (1000, 513, 129),  # 32 x 32
         (2048, 1024, 96), (1477, 1477, 37),  # 64 x 64
         (4096, 2048, 48), (4099, 2051, 17)]  # (more of them: 128 x 128 ones take contractions of 256 and more)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_tiles(L, M, N, K, layout):
    product(L, M, N, K, layout, epilogue=(M + K) % 2 == 1)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("odd", [1, 2, 3])
def test_rows_at_any_element(L, layout, odd):
    product(L, 131, 78, 83, layout, odd=odd)
    product(L, 1477, 1474, 33, layout, odd=odd)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(77, 64, 50), (256, 256, 64), (130, 257, 33)])
def test_batches(L, M, N, K, layout):
    product(L, M, N, K, layout, batch=(3, 5))
    product(L, M, N, K, layout, batch=(31, 1))
