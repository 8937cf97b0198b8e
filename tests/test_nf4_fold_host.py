"""NF4-coded products that take an adapter's update inside them: what the planner makes of a step with them, and that
its launches (on the host interpreter of the launch records) round where they did without."""
import numpy as np
import pytest
import torch

import nabla_amd as nb
from nabla_amd.core import engine

BF16 = nb.DType.bfloat16
LEVELS = torch.from_numpy(np.asarray(nb.nn.finetune.qlora.NF4_CODEBOOK, np.float32))


class Pair:
    """A weight as codes, an adapter and rows to multiply, with their float64 values."""

    def __init__(self, tokens, rows, cols, rank, seed=0):
        gen = torch.Generator().manual_seed(seed + rows)
        self.codes = torch.randint(0, 16, (rows * cols,), generator=gen, dtype=torch.uint8)
        self.scales = torch.rand(rows * cols // 64, generator=gen) * 0.2
        self.x, self.a, self.b = ((torch.randn(s, generator=gen) * std).to(torch.bfloat16)
                                  for s, std in (((tokens, rows), 1.0), ((rows, rank), 0.1), ((rank, cols), 0.5)))
        self.weight = dict(indices=nb.Tensor.from_dlpack(self.codes), scales=nb.Tensor.from_dlpack(self.scales),
                           original_shape=(rows, cols), original_numel=rows * cols, padded_numel=rows * cols, block_size=64)
        self.adapter = {"A": nb.Tensor.from_dlpack(self.a), "B": nb.Tensor.from_dlpack(self.b)}

    def linear(self, x, adapter=None):
        return nb.nn.finetune.qlora_linear(x, self.weight, adapter or self.adapter, alpha=float(self.a.shape[1]), compute_dtype=BF16)

    def exact(self):
        w = (LEVELS[self.codes.long()].view(-1, 64) * self.scales[:, None]).view(self.x.shape[1], -1).to(torch.bfloat16)
        thin = (self.x.double() @ self.a.double()).to(torch.bfloat16).double()  # (a product of its own: stored)
        return self.x.double() @ w.double() + thin @ self.b.double()


def planned(*outputs):
    engine.clear_plan_cache()
    nb.realize_all(*outputs)
    steps = [s for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps]
    engine.clear_plan_cache()
    return steps


def folded(steps):
    return [s for s in steps if s.kind == "gemm_nf4" and s.attrs.get("terms")]


def test_a_function_of_the_sum_is_of_the_sum_before_it_is_rounded(emulator):
    p = Pair(160, 128, 192, 8)
    pre = p.linear(nb.Tensor.from_dlpack(p.x))
    h = nb.gelu(pre)
    steps = planned(pre, h)
    assert len(folded(steps)) == 1 and not any(s.kind == "gemm" and s.attrs["K"] == 8 for s in steps)
    want = p.exact()
    # (each output rounded once, half a unit of eight bits, behind sums in float32)
    for got, exact in ((pre, want), (h, torch.nn.functional.gelu(want))):
        assert ((got.to_torch().double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 2e-5).all()


def test_a_sum_that_nothing_computes_on_is_rounded_by_its_product(emulator):
    p = Pair(160, 128, 192, 8)
    pre = p.linear(nb.Tensor.from_dlpack(p.x))
    steps = planned(pre)
    assert [s.attrs["dst"].dtype for s in folded(steps)] == [BF16] and not any(s.kind == "rowprog" for s in steps)
    assert ((pre.to_torch().double() - p.exact()).abs() <= 2.0 ** -8 * p.exact().abs() + 2e-5).all()


@pytest.mark.parametrize("tokens,rows,cols,rank,inside", [
    (128, 128, 128, 8, 1), (127, 128, 128, 8, 0), (128, 64, 128, 8, 0), (128, 192, 128, 64, 1), (128, 160, 128, 8, 0),
    (128, 128, 64, 8, 0), (128, 128, 192, 72, 0), (128, 128, 192, 4, 0)])
def test_where_the_update_goes_inside(emulator, tokens, rows, cols, rank, inside):
    """From 128 rows, columns and numbers of a sum on, for contractions of whole K tiles and ranks of whole chunks up to one."""
    p = Pair(tokens, rows, cols, rank)
    y = p.linear(nb.Tensor.from_dlpack(p.x))
    steps = planned(y)
    assert len(folded(steps)) == inside
    # (a sum that is no part of the product: base and update rounded by themselves, and what they come to)
    size = p.exact().abs() + 2.0 * (p.x.double().abs() @ p.a.double().abs()) @ p.b.double().abs()
    assert ((y.to_torch().double() - p.exact()).abs() <= 2.0 ** (-8 if inside else -7) * size + 2e-5).all()


def test_an_update_that_is_used_twice_stays_a_product(emulator):
    p = Pair(160, 128, 192, 8)
    x = nb.Tensor.from_dlpack(p.x)
    base = p.linear(x, {k: nb.zeros_like(v) for k, v in p.adapter.items()})
    thin = (x @ p.adapter["A"]) @ p.adapter["B"]
    steps = planned(base + thin, thin)
    assert not any(t["K"] == 8 and s.attrs["N"] != 192 for s in folded(steps) for t in s.attrs["terms"])
    assert any(s.kind == "gemm" and s.attrs["N"] == 192 for s in steps)
