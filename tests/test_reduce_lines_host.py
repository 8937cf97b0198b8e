"""Sums of numbers that lie behind each other: how many of them the planner leaves to one launch."""
import numpy as np
import pytest
import torch

import nabla_amd as nb
from nabla_amd.core import engine


@pytest.mark.parametrize("dtype,n,first,launches", [
    ("float32", 65536, 0, 1), ("float32", 65600, 0, 2), ("bfloat16", 65536, 0, 1), ("bfloat16", 65536, 8, 1),
    # behind an odd element, or of no whole 16 bytes: by element
    ("float32", 16384, 1, 2), ("bfloat16", 16384, 4, 2), ("float32", 8192, 1, 1), ("float32", 8190, 0, 1), ("float32", 16386, 0, 2),
    ("float16", 4096, 0, 1), ("float16", 8192, 0, 2), ("float16", 65536, 0, 2)])
def test_one_launch_or_two(emulator, dtype, n, first, launches):
    x = torch.tensor(np.random.default_rng(n).integers(-2, 3, n + 8).astype(np.float32)).to(getattr(torch, dtype))
    engine.clear_plan_cache()
    y = nb.reduce_sum(nb.reshape(nb.Tensor.from_dlpack(x)[first:first + n], (n, 1)), axis=0, keepdims=True)
    nb.realize_all(y)
    steps = [s for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps]
    engine.clear_plan_cache()
    assert [s.kind for s in steps] == ["reduce_mid"] * launches
    want = x[first:first + n].double().sum()
    assert abs(float(y.to_torch().double()) - want) <= 2.0 ** -8 * abs(want)
