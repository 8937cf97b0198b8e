"""Reductions whose results a later step of the plan reads go out together; with no room to wait each
goes out by itself, which is the reference here."""
import numpy as np
import pytest

import nabla_amd as nb
from nabla_amd.backend.planner import Planner
from nabla_amd.core import engine
from nabla_amd.nn import optim


def T(a, dtype=nb.DType.float32):
    return nb.Tensor.constant(np.asarray(a, dtype=np.float32), dtype=dtype)


def both_ways(monkeypatch, make):
    """(results, launches of reductions) with room to wait and without."""
    out = []
    for room in (Planner.MAX_WAITING_BYTES, -1):
        monkeypatch.setattr(Planner, "MAX_WAITING_BYTES", room)
        engine.clear_plan_cache()
        got = [nb.cast(t, nb.DType.float32).numpy() for t in make()]
        out.append((got, sum(s.kind in ("reduce_mid", "reduce_batch")
                             for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps)))
    engine.clear_plan_cache()
    return out


@pytest.mark.parametrize("dtype", [nb.DType.float32, nb.DType.bfloat16])
@pytest.mark.parametrize("rows", [1, 40, 1600, 8200])
def test_bias_gradients_that_an_update_reads(emulator, monkeypatch, rows, dtype):
    rng = np.random.default_rng(rows)
    sizes = (24, 64, 40, 64)
    w = [rng.standard_normal((a, b)) * a ** -0.5 for a, b in zip(sizes, sizes[1:])]
    b = [rng.standard_normal(n) for n in sizes[1:]]
    x = rng.standard_normal((rows, sizes[0]))

    def make():
        params = [T(a, dtype) for a in w + b]

        def loss(*p):
            h = T(x, dtype)
            for i in range(3):
                h = nb.relu(h @ p[i] + p[3 + i])
            return nb.reduce_sum(nb.cast(h * h, nb.DType.float32))

        def step(*p):
            grads = nb.grad(loss, argnums=tuple(range(6)))(*p)
            new, state = optim.adamw_update(list(p), list(grads), optim.adamw_init(list(p)), lr=0.01)
            return list(grads) + new

        return nb.compile(step)(*params)

    (got, n), (want, n_alone) = both_ways(monkeypatch, make)
    # (in bf16 the sums ride on the products of the weight gradients, which are next in the plan)
    assert n < n_alone or (n == n_alone and (rows == 1 or dtype is nb.DType.bfloat16))
    for a, c in zip(got[:6], want[:6]):
        # the same sums in the same order; column sums that ride on a bf16 product are added in its
        # order: two float32 sums of rows terms, and one rounding to bf16 each of them
        tol = 0 if dtype is nb.DType.float32 else 2.0 ** -7
        np.testing.assert_allclose(a, c, rtol=tol, atol=tol)


def test_fused_groups_that_read_waiting_results(emulator, monkeypatch):
    """A chain over more results than one row program takes."""
    rng = np.random.default_rng(0)
    mats = [rng.standard_normal((7, 5, 48)) for _ in range(30)]

    def make():
        def f(*m):
            out = 0.0
            for a in m:
                out = nb.sin(out + nb.reduce_sum(a, axis=1))
            return [out]
        return nb.compile(f)(*[T(a) for a in mats])

    (got, n), (want, n_alone) = both_ways(monkeypatch, make)
    assert n < n_alone
    np.testing.assert_array_equal(got[0], want[0])


def test_sources_above_the_limit_do_not_wait(emulator, monkeypatch):
    """x @ w, its column sums, and six products before a step reads them: a source larger than the limit is
    reduced behind the product that writes it, and its memory is free for the next one."""
    rng = np.random.default_rng(0)
    w = [rng.standard_normal((256, 256)) for _ in range(7)]
    x = rng.standard_normal((512, 256))

    def make():
        def f(x, *w):
            x = x @ w[0]
            total = nb.reduce_sum(x, axis=0)
            for m in w[1:]:
                x = x @ m
            return [total + x]
        return nb.compile(f)(T(x), *[T(m) for m in w])

    plans = {}
    for limit in (Planner.MAX_WAITING_BYTES, x.nbytes // 2 - 1, -1):  # (x is float64: half of it in float32)
        monkeypatch.setattr(Planner, "MAX_WAITING_BYTES", limit)
        engine.clear_plan_cache()
        got = make()[0].numpy()
        (plan,) = [bp.plan for bp in engine._PLAN_CACHE.values()]
        kinds = [s.kind for s in plan.steps]
        plans[limit] = (kinds.index("reduce_mid"), plan.arena_bytes, got)
    engine.clear_plan_cache()
    (at_wait, arena_wait, want), (at, arena, got), (at_never, arena_never, _) = plans.values()
    assert at_wait == 6 and at == at_never == 1
    assert arena == arena_never < arena_wait
    np.testing.assert_array_equal(got, want)


def test_all_that_wait_together_stay_below_the_limit(emulator, monkeypatch):
    """Three sources at the limit wait for their reader; where two fit, the third sends the first two out."""
    rng = np.random.default_rng(0)
    x = rng.standard_normal((64, 128))
    w = [rng.standard_normal((128, 128)) for _ in range(4)]

    def make():
        def f(x, *w):
            sums = 0.0
            for m in w[:3]:
                x = x @ m
                sums = nb.sin(sums + nb.reduce_sum(x, axis=0))
            return [sums + x @ w[3]]
        return nb.compile(f)(T(x), *[T(m) for m in w])

    for fit, launches in ((3, ["reduce_batch"]), (2, ["reduce_batch", "reduce_mid"])):
        monkeypatch.setattr(Planner, "MAX_WAITING_BYTES", fit * 64 * 128 * 4)
        engine.clear_plan_cache()
        make()
        (plan,) = [bp.plan for bp in engine._PLAN_CACHE.values()]
        engine.clear_plan_cache()
        assert [s.kind for s in plan.steps if s.kind.startswith("reduce")] == launches
