"""Products with NF4-coded weights that decode into a workspace, where the block length, the last
workgroup of the decoder, the contraction's length and the row stride can go wrong: against
float64 on the weight the oracle decodes (rounded to bf16 once for bf16), and the fused kernel."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ops as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("transpose", [0, 1])
@pytest.mark.parametrize("M,rows,cols,block,lda", [(1, 128, 128, 64, 0), (77, 136, 200, 8, 3), (300, 1000, 264, 24, 0),
                                                   (520, 512, 1024, 64, 8), (33, 64, 72, 8, 0)])
def test_decoded_product(M, rows, cols, block, lda, transpose, dtype):
    from nabla_amd.backend import lib
    rng = np.random.default_rng(rows + cols)
    q = O.nf4_quantize(rng.standard_normal((rows, cols)).astype(np.float32), block)
    w = torch.tensor(O.nf4_dequantize(q)).to(dtype).double()
    K, N = (cols, rows) if transpose else (rows, cols)
    x = torch.zeros(M, K + lda, dtype=dtype)
    x[:, :K] = torch.tensor(rng.standard_normal((M, K)))
    want = x[:, :K].double() @ (w.t() if transpose else w)
    xd, codes, scales = x.cuda(), torch.tensor(q["indices"]).cuda(), torch.tensor(q["scales"]).cuda()
    out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    size = rows * cols * dtype.itemsize
    ws = torch.full((rows * cols + 64,), 7.0, dtype=dtype, device="cuda")
    d = lib.GemmNf4Desc()
    d.A, d.codes, d.scales, d.C = xd.data_ptr(), codes.data_ptr(), scales.data_ptr(), out.data_ptr()
    d.M, d.w_rows, d.w_cols, d.lda, d.ldc = M, rows, cols, K + lda, N
    d.block, d.transpose_w, d.dtype, d.alpha = block, transpose, (1 if dtype is torch.bfloat16 else 0), 1.0
    d.workspace, d.workspace_bytes = ws.data_ptr(), size
    L = lib.load()
    lib.check(L.nbk_gemm_nf4(C.byref(d), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    # one rounding of the result; float32 sums of K terms stay well inside K^(1/2) roundings
    rtol, atol = (2.0 ** -8, 1e-4) if dtype is torch.bfloat16 else (1e-6, 6e-8 * K)
    err = (out.double().cpu() - want).abs() - rtol * want.abs()
    assert err.max().item() <= atol * want.abs().max().item()
    if K >= 128:
        assert torch.equal(ws[:rows * cols].cpu().double(), w.reshape(-1))
        d.workspace_bytes = size - 1
        with pytest.raises(ValueError, match="workspace"):
            lib.check(L.nbk_gemm_nf4(C.byref(d), None))
    assert (ws[rows * cols:] == 7).all()
