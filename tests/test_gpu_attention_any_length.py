"""Fused attention over sequences that are no multiple of the 128-row tiles: a handful of tokens,
one short of and one past a tile of 64 and of 128, and several tiles with a rest, against float64."""
import numpy as np
import pytest
import torch

import nabla_amd as nb

pytestmark = pytest.mark.gpu


# bf16 inputs and results: a result is rounded once (2^-9 of its size) and the probabilities once
# before the second product; gradients pass through two such products.  2e-2 of the largest value
# of a tensor is the bound the aligned lengths are held to.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("b,h,s,hd", [(2, 3, 1, 64), (1, 2, 5, 128), (2, 2, 63, 64), (1, 3, 65, 128), (1, 2, 127, 64),
                                      (2, 1, 129, 64), (1, 2, 200, 128), (1, 2, 333, 64), (1, 1, 333, 128),
                                      (1, 1, 1100, 64)])
def test_any_length(hip, b, h, s, hd, causal):
    gen = torch.Generator().manual_seed(s * 2 + causal)
    shape = (b, s, h * hd)  # (heads are read in place out of wider rows)
    q, k, v, g = (torch.randn(shape, generator=gen).to(torch.bfloat16) for _ in range(4))
    x = [nb.Tensor.from_dlpack(t.cuda()) for t in (q, k, v, g)]

    def heads(t):
        return nb.swap_axes(nb.reshape(t, (b, s, h, hd)), 1, 2)

    def loss(q, k, v):
        o = nb.nn.functional.scaled_dot_product_attention(heads(q), heads(k), heads(v), is_causal=causal)
        o = nb.reshape(nb.swap_axes(o, 1, 2), shape)
        return nb.reduce_sum(nb.cast(o * x[3], nb.DType.float32)), o

    print("attention", (b, h, s, hd), causal, flush=True)
    out = loss(*x[:3])[1]
    grads = nb.grad(lambda *a: loss(*a)[0], argnums=(0, 1, 2))(*x[:3])
    nb.realize_all(out, *grads)
    from nabla_amd.core import engine
    plans = [p.plan.stats for p in engine._PLAN_CACHE.values()]
    assert any(st.get("attention") and st.get("attention_bwd") for st in plans)

    leaf = [t.double().requires_grad_() for t in (q, k, v)]
    split = [t.reshape(b, s, h, hd).transpose(1, 2) for t in leaf]
    score = split[0] @ split[1].transpose(-1, -2).contiguous() / hd ** 0.5
    if causal:
        score = score.masked_fill(~torch.ones(s, s, dtype=torch.bool).tril(), float("-inf"))
    want = (torch.softmax(score, -1) @ split[2]).transpose(1, 2).reshape(shape)
    (want * g.double()).sum().backward()
    scale = max(t.grad.abs().max().item() for t in leaf)
    for got, ref in zip([out, *grads], [want.detach(), *(t.grad for t in leaf)]):
        err = (got.to_torch().double().cpu() - ref).abs().max().item()
        # (dq and dk of a single visible key are zero: measured against the other gradients)
        assert err <= 2e-2 * max(ref.abs().max().item(), 0.05 * scale)
