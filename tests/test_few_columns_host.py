"""bf16 products with few columns: the planner keeps one whole where the launch takes the kernel that splits K over a
workgroup's waves, and nowhere else for that reason."""
import ctypes as C
import random

import pytest
import torch

import nabla_amd as nb
from nabla_amd.backend import lib
from nabla_amd.backend.planner import Planner
from nabla_amd.core import engine


def test_both_sides_ask_the_same():
    rng, L, taken = random.Random(0), lib.load(), 0
    rows = [1, 15, 16, 17, 200, 1000, 1023, 1024, 4000, 8191, 8192, 8193, 20000]
    for _ in range(20000):
        M, N = rng.choice(rows), rng.choice([1, 2, 4, 7, 8, 10, 12, 16, 20, 24, 31, 32, 33, 40])
        K = rng.choice([64, 128, 192, 256, 320, 1000, 1024, 1984, 2048, 2112, 4032, 4096, 4160, 8128, 8192])
        lda, off_a, off_b = K + rng.choice([0, 0, 0, 4, 8]), rng.choice([0, 0, 0, 8, 1]), rng.choice([0, 0, 0, 16, 4])
        pa = ((), lda, 1)
        pb = ((), 1, K + rng.choice([0, 0, 8, 2])) if rng.random() < 0.5 else ((), N + rng.choice([0, 0, 3, 8]), 1)
        d = lib.GemmDesc()
        d.A, d.B, d.C = 4096 + 2 * off_a, 4096 + 2 * off_b, 4096
        d.M, d.N, d.K, d.a_rs, d.a_cs, d.b_rs, d.b_cs, d.ldc = M, N, K, pa[1], 1, pb[1], pb[2], N
        d.batch, d.batch_inner, d.dtype_ab, d.dtype_c, d.alpha = 1, 1, 1, 1, 1.0
        got = L.nbk_gemm_few_columns(C.byref(d))
        assert got == Planner._few_columns(M, N, K, pa, pb, off_a, off_b), (M, N, K, pa, pb, off_a, off_b)
        taken += got
    assert taken > 1000


def slices(M, N, K, view=None):
    gen = torch.Generator().manual_seed(N)
    a, b = (torch.randn(s, generator=gen).to(torch.bfloat16) for s in ((M, K + 8), (K, N)))
    x, w = nb.Tensor.from_dlpack(a), nb.Tensor.from_dlpack(b)
    engine.clear_plan_cache()
    y = (x[:, 1:K + 1] if view == "odd" else x[:, :K]) @ w
    nb.realize_all(y)
    steps = [s for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps if s.kind == "gemm"]
    engine.clear_plan_cache()
    rows = a[:, 1:K + 1] if view == "odd" else a[:, :K]
    want = rows.double() @ b.double()
    assert (y.to_torch().double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    return [s.attrs["batch"] for s in steps]


@pytest.mark.parametrize("M", [16, 64, 200, 1000])
@pytest.mark.parametrize("N,K,want", [(4, 2048, 4), (12, 1024, 2), (20, 2048, 4), (10, 1920, 2), (8, 2048, 1), (16, 2048, 1),
                                      (32, 1024, 1)])
def test_what_that_kernel_refuses_stays_in_slices(emulator, M, N, K, want):
    assert slices(M, N, K) == [want]


def test_rows_of_no_whole_chunks_stay_in_slices(emulator):
    assert slices(200, 8, 2048) == [1] and slices(200, 8, 2048, view="odd") == [4]
