"""An NF4-coded product with an adapter's update inside it, both orientations, out of a workspace and without one,
against the decoded weight in float64."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transpose", [0, 1])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("M,rows,cols,ranks", [(1000, 256, 640, (8,)), (128, 128, 128, (64,)), (200, 192, 320, (16, 8)), (77, 64, 136, (8,)),
                                               (300, 320, 192, (5,))])
def test_update_inside(hip, M, rows, cols, ranks, workspace, dtype, transpose):
    import nabla_amd as nb
    from nabla_amd.backend import lib
    t = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(M + rows + cols)
    K, N = (cols, rows) if transpose else (rows, cols)
    block = 8 if rows * cols % 64 else 64
    codes = torch.randint(0, 16, (rows * cols,), generator=gen, device="cuda").to(torch.uint8)
    scales = torch.rand(rows * cols // block, generator=gen, device="cuda") + 0.5
    level = torch.from_numpy(np.asarray(nb.nn.finetune.qlora.NF4_CODEBOOK, np.float32)).cuda()
    w = (level[codes.long()].view(-1, block) * scales[:, None]).view(rows, cols)
    w = w.to(t).double()
    w = w.t().contiguous() if transpose else w
    x = torch.randn(M, K, generator=gen, device="cuda").to(t)
    out = torch.full((M, N), float("nan"), dtype=t, device="cuda")
    ws = torch.empty(rows * cols, dtype=t, device="cuda")
    d = lib.GemmNf4Desc()
    d.A, d.codes, d.scales, d.C = x.data_ptr(), codes.data_ptr(), scales.data_ptr(), out.data_ptr()
    d.M, d.w_rows, d.w_cols, d.lda, d.ldc, d.block, d.transpose_w = M, rows, cols, K, N, block, transpose
    d.dtype, d.alpha = (1 if dtype == "bfloat16" else 0), 1.0
    if workspace:
        d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel() * ws.element_size()
    want, size = x.double() @ w, x.double().abs() @ w.abs()
    terms, keep = (lib.GemmTerm * len(ranks))(), []
    for p, r in zip(terms, ranks):
        u, v = (torch.randn(s, generator=gen, device="cuda").to(t) for s in ((M, r), (r, N)))
        stored = v.t().contiguous() if transpose else v
        keep += [u, stored]
        p.A, p.B, p.K, p.a_rs, p.a_cs = u.data_ptr(), stored.data_ptr(), r, r, 1
        p.b_rs, p.b_cs = (1, r) if transpose else (N, 1)
        want += u.double() @ v.double()
        size += u.double().abs() @ v.double().abs()
    lib.check(lib.load().nbk_gemm_nf4_terms(C.byref(d), terms, len(ranks), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    # sums in float32 (2^-22 of all that is added covers K of 640); a bf16 result is rounded once for the product and
    # once more for each pair that does not go inside it
    rounds = (2.0 ** -9 * (1 + len(ranks)) if dtype == "bfloat16" else 0.0)
    assert ((out.double() - want).abs() <= 2.0 ** -20 * size + rounds * size.clamp(min=1e-6).minimum(want.abs() + 2.0 ** -1 * size)).all()


@pytest.mark.parametrize("transpose", [0, 1])
@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("M,rows,cols,rank", [(1000, 256, 640, 8), (129, 128, 136, 64), (77, 64, 136, 8), (300, 320, 192, 5)])
def test_float32_result_of_bf16_operands(hip, M, rows, cols, rank, workspace, transpose):
    """Nothing is rounded to bf16 but the operands."""
    import nabla_amd as nb
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(M + cols)
    K, N = (cols, rows) if transpose else (rows, cols)
    codes = torch.randint(0, 16, (rows * cols,), generator=gen, device="cuda").to(torch.uint8)
    scales = torch.rand(rows * cols // 64, generator=gen, device="cuda") + 0.5
    level = torch.from_numpy(np.asarray(nb.nn.finetune.qlora.NF4_CODEBOOK, np.float32)).cuda()
    w = (level[codes.long()].view(-1, 64) * scales[:, None]).view(rows, cols).to(torch.bfloat16).double()
    w = w.t().contiguous() if transpose else w
    x, u, v = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16) for s in ((M, K), (M, rank), (rank, N)))
    stored = v.t().contiguous() if transpose else v
    out, ws = torch.full((M, N), float("nan"), device="cuda"), torch.empty(rows * cols, dtype=torch.bfloat16, device="cuda")
    d = lib.GemmNf4Desc()
    d.A, d.codes, d.scales, d.C = x.data_ptr(), codes.data_ptr(), scales.data_ptr(), out.data_ptr()
    d.M, d.w_rows, d.w_cols, d.lda, d.ldc, d.block, d.transpose_w, d.dtype, d.alpha = M, rows, cols, K, N, 64, transpose, 1, 1.0
    if workspace:
        d.workspace, d.workspace_bytes = ws.data_ptr(), 2 * ws.numel()
    terms = (lib.GemmTerm * 1)()
    terms[0].A, terms[0].B, terms[0].K, terms[0].a_rs, terms[0].a_cs = u.data_ptr(), stored.data_ptr(), rank, rank, 1
    terms[0].b_rs, terms[0].b_cs = (1, rank) if transpose else (N, 1)
    lib.check(lib.load().nbk_gemm_nf4_terms_f32(C.byref(d), terms, 1, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    size = x.double().abs() @ w.abs() + u.double().abs() @ v.double().abs()
    # (704 exact products at most, added in float32: 2^-24 of all that is added for each of up to 16 steps of a chain)
    assert ((out.double() - (x.double() @ w + u.double() @ v.double())).abs() <= 2.0 ** -20 * size).all()
