"""Products x^T dy split along a contraction that no number of slices divides: every slice lies inside
the operands and the slices cover them once."""
import numpy as np
import pytest

import nabla_amd as nb
from nabla_amd.core import engine


def bf16(a):
    return nb.Tensor.constant(a, dtype=nb.DType.bfloat16)


def check_slices(a, K):
    """The K range of every member of a launch, against the rule of ``nbk_gemm_desc.k_last``."""
    ks = a["batch_inner"] if a["batch_inner"] > 1 else a["batch"]
    assert 0 <= a["k_last"] < a["K"] and (ks - 1) * a["K"] + (a["k_last"] or a["K"]) == K


# (rounded up to whole tiles of 64, sixteen and more slices can cover K before the last one)
@pytest.mark.parametrize("M,N,K", [(512, 512, 8200), (512, 512, 9600), (256, 256, 8640), (16, 16, 16400),
                                   (2048, 16, 9216), (64, 24, 33000)])
def test_a_weight_gradient_over_many_rows(emulator, M, N, K):
    rng = np.random.default_rng(K)
    x, g = rng.integers(-2, 3, (K, M)).astype(np.float32), rng.integers(-2, 3, (K, N)).astype(np.float32)
    engine.clear_plan_cache()
    got = nb.grad(lambda w: nb.reduce_sum(nb.cast((bf16(x) @ w) * bf16(g), nb.DType.float32)))(
        bf16(np.zeros((M, N), np.float32)))
    got = nb.cast(got, nb.DType.float32).numpy()
    launches = [s.attrs for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps
                if s.kind == "gemm" and s.attrs["batch"] > 1]
    assert len(launches) == 1
    check_slices(launches[0], K)
    want = x.T @ g  # (whole numbers, exact in float32; the result is rounded to bf16 once)
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want)).all()
    engine.clear_plan_cache()


def test_joined_projections_over_many_rows(emulator):
    """The gradients of three projections of one input, members of one launch."""
    K, d, heads = 8640, 64, 1
    rng = np.random.default_rng(3)
    x = bf16(rng.standard_normal((8, K // 8, d)).astype(np.float32))
    w = [bf16(rng.standard_normal((d, d)).astype(np.float32) * d ** -0.5) for _ in range(3)]

    def loss(*w):
        q, k, v = (nb.swap_axes(nb.reshape(x @ u, (8, K // 8, heads, d)), 1, 2) for u in w)
        o = nb.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True)
        return nb.mean(nb.cast(o * o, nb.DType.float32))

    engine.clear_plan_cache()
    grads = nb.grad(loss, argnums=(0, 1, 2))(*w)
    nb.realize_all(*grads)
    launches = [s.attrs for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps
                if s.kind == "gemm" and s.attrs["batch"] > 1]
    assert any(a["batch_inner"] > 1 for a in launches)
    for a in launches:
        check_slices(a, K)
    engine.clear_plan_cache()


def test_every_contraction_length():
    from nabla_amd.backend.planner import Planner
    for M, N in [(8, 8), (256, 256), (512, 512), (2048, 16), (1024, 1024), (1024, 4096)]:
        for K in list(range(1024, 20000)) + list(range(20000, 70000, 7)):
            ks = Planner._split_k(M, N, K, nb.DType.bfloat16, rows_contiguous=True)
            if ks > 1:
                n, kc, last = Planner._slices(K, ks)
                assert kc % 64 == 0 and 2 <= n <= ks and (n - 1) * kc < K <= n * kc, (M, N, K)
                assert last == (0 if n * kc == K else K - (n - 1) * kc), (M, N, K)


def test_a_last_slice_longer_than_the_others_is_refused():
    """On the host, before anything is launched: it would be read from behind the operands."""
    import ctypes as C
    from nabla_amd.backend import lib
    L = lib.load()
    for dtype, k_last, batch in [(1, 65, 4), (0, 65, 4), (1, 1 << 30, 1), (1, -1, 4)]:
        d = lib.GemmDesc()
        d.A = d.B = d.C = 4096
        d.M = d.N = d.K = 64
        d.a_rs, d.a_cs, d.b_rs, d.b_cs, d.ldc = 1, 64, 64, 1, 64
        d.batch, d.batch_inner, d.a_bs, d.b_bs, d.c_bs = batch, 1, 4096, 4096, 4096
        d.dtype_ab, d.dtype_c, d.alpha, d.k_last = dtype, 0, 1.0, k_last
        with pytest.raises(ValueError, match="k_last"):
            lib.check(L.nbk_gemm(C.byref(d), None))


def test_few_workgroups_and_a_middling_contraction_are_split():
    """Results of 33 to 256 tiles of 64 x 64 wait for one workgroup's loop over K: whole, 512 x 512 x
    3072 takes twice what it takes in four slices.  What can be folded into the product outweighs
    that up to 2048."""
    from nabla_amd.backend.planner import Planner
    for kind in (dict(rows_contiguous=True), dict(a_k_contiguous=True)):
        def split(M, N, K, **kw):
            return Planner._split_k(M, N, K, nb.DType.bfloat16, **kind, **kw)
        assert split(512, 512, 1024) == 1
        assert split(512, 512, 1536) == 2 and split(1024, 1024, 1536) == 2
        assert split(512, 512, 2048) == 4 and split(512, 512, 3072) == 4
        assert split(768, 768, 2048) == 4 and split(1024, 1024, 3072) == 2
        assert split(512, 512, 4096) == 8 and split(512, 1024, 4096) == 4
        assert split(1024, 1536, 2048) == 1 and split(1792, 1024, 4096) == 1
        assert split(512, 512, 2048, epilogue=True) == 1 and split(512, 512, 3072, epilogue=True) == 4
    assert Planner._split_k(512, 512, 1998, nb.DType.bfloat16, rows_contiguous=True) == 2
    assert Planner._split_k(512, 512, 1998, nb.DType.bfloat16, a_k_contiguous=True) == 1
