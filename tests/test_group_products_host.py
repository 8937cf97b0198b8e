"""Products x^T dy that go out together: which do, in which order everything runs then, and that what they use stays in
memory until their launch."""
import numpy as np
import pytest

import nabla_amd as nb
from nabla_amd.backend.planner import Buf, Planner, Step, ViewRef
from nabla_amd.core import engine
from nabla_amd.core.dtype import DType


# ---- the reordering by itself ------------------------------------------------------------------
def ref(buf):
    return ViewRef(buf, 0, (64, 64), (64, 1), DType.float32)


def product(a, b, dst, **attrs):
    return Step("gemm", [a, b], [dst], dict(dict(a=ref(a), b=ref(b), dst=ref(dst), M=64, N=64, K=64, a_rs=1, a_cs=64, b_rs=64,
                                                 b_cs=1, batch=1), **attrs))


def other(reads, writes):
    return Step("copy", list(reads), list(writes))


def reordered(*steps):
    """Names of the steps as they run (a group in brackets), and the live ranges of the buffers."""
    p = Planner.__new__(Planner)
    p.steps = list(steps)
    n = 1 + max(b for s in steps for b in s.reads + s.writes)
    p.bufs = [Buf(i, 4096, DType.float32, "temp") for i in range(n)]
    for i, s in enumerate(steps):
        for b in s.reads + s.writes:
            p.bufs[b].first, p.bufs[b].last = min(p.bufs[b].first, i), max(p.bufs[b].last, i)
    p._group_products()
    order = [next(i for i, s in enumerate(steps) if s is t) for t in p.steps]
    groups = [p.steps[k].attrs.get("group") for k in range(len(order))]
    return order, groups, {b.id: (b.first, b.last) for b in p.bufs}


def test_a_product_moves_to_the_last_of_its_group():
    order, groups, live = reordered(product(0, 1, 2), other([1], [3]), product(0, 3, 4), other([2, 4], [5]))
    assert order == [1, 0, 2, 3] and groups == [None, 1, 1, None]
    # (both run at once: what either uses is there from the first to the last of them)
    assert live[1] == (0, 2) and live[0] == (1, 2) and live[3] == (0, 2) and live[2] == live[4] == (1, 3)


@pytest.mark.parametrize("between", [other([2], [5]), other([6], [0]), other([6], [1]), other([6], [2])],
                         ids=["reads the result", "overwrites an operand", "overwrites the other", "overwrites the result"])
def test_what_meets_a_waiting_product_ends_its_group(between):
    order, groups, _ = reordered(product(0, 1, 2), between, product(7, 3, 4))
    assert order == [0, 1, 2] and groups == [None] * 3


@pytest.mark.parametrize("second", [product(2, 1, 4), product(7, 3, 0), product(7, 3, 2), product(0, 3, 4, M=64 * 513),
                                    product(7, 3, 4, a_cs=1), product(7, 3, 4, b_rs=1), product(7, 3, 4, K=1),
                                    product(7, 3, 4, bias=ref(8)), product(7, 3, 4, members=[1])],
                         ids=["reads the first", "overwrites its operand", "overwrites its result", "large", "A in rows",
                              "B in columns", "one number", "bias", "members"])
def test_products_that_do_not_join(second):
    order, groups, _ = reordered(product(0, 1, 2), second)
    assert order == [0, 1] and groups == [None, None]


def test_a_group_ends_at_seven_and_at_the_window():
    order, groups, _ = reordered(*[product(0, 1, 2 + i) for i in range(9)])
    assert order == list(range(9)) and groups == [1] * 7 + [2] * 2
    steps = [product(0, 1, 2)] + [other([3], [3]) for _ in range(24)] + [product(0, 1, 4)]
    assert reordered(*steps)[1] == [None] * 26
    assert reordered(*steps[:24], steps[-1])[1] == [None] * 23 + [1, 1]


# ---- in plans ------------------------------------------------------------------------------------
def layers(dtype, optimizer, bias=True):
    rng = np.random.default_rng(3)

    def T(*shape):
        return nb.cast(nb.Tensor.constant(rng.standard_normal(shape).astype(np.float32) * 0.3), dtype)

    sizes = [64, 256, 128, 256, 64]
    params = [(T(a, b), T(1, b)) for a, b in zip(sizes, sizes[1:])]
    x = T(2048 if dtype is DType.bfloat16 else 256, 64)

    def loss(params, x):
        for w, b in params:
            x = nb.gelu(x @ w + b if bias else x @ w) + nb.mean(x)
        return nb.mean(x * x)

    nb.realize_all(x, *nb.tree_leaves(params))
    engine.clear_plan_cache()
    value, grads = nb.value_and_grad(loss)(params, x)
    out = [value, *nb.tree_leaves(grads)]
    if optimizer:
        state = nb.nn.optim.adamw_init(params)
        out = nb.tree_leaves(nb.nn.optim.adamw_update(params, grads, state, lr=1e-3, realize=False))
    nb.realize_all(*(t for t in out if isinstance(t, nb.Tensor)))
    plan = max((bp.plan for bp in engine._PLAN_CACHE.values()), key=lambda p: len(p.steps))
    engine.clear_plan_cache()
    return plan, [nb.cast(t, DType.float32).numpy() for t in out if isinstance(t, nb.Tensor)]


@pytest.mark.parametrize("dtype", [DType.float32, DType.bfloat16], ids=["float32", "bfloat16"])
@pytest.mark.parametrize("optimizer", [False, True])
def test_buffers_of_a_group_live_until_its_launch(emulator, monkeypatch, dtype, optimizer):
    plan, got = layers(dtype, optimizer)
    grouped = [s for s in plan.steps if "group" in s.attrs]
    assert len(grouped) >= 3
    if dtype is DType.bfloat16:  # (slices of K and column sums too)
        assert any(s.attrs["batch"] > 1 for s in grouped) and any(s.attrs.get("colsum") is not None for s in grouped)
    instant, at = {}, -1  # (members of a group run at one)
    for k, s in enumerate(plan.steps):
        if not (k and "group" in s.attrs and s.attrs["group"] == plan.steps[k - 1].attrs.get("group")):
            at += 1
        instant[k] = at
    live = {}
    for k, s in enumerate(plan.steps):
        for b in s.reads + s.writes:
            lo, hi = live.get(b, (instant[k], instant[k]))
            live[b] = (min(lo, instant[k]), max(hi, instant[k]))
    temps = [b for b in plan.bufs if b.role == "temp" and b.id in live]
    for i, b in enumerate(temps):
        for c in temps[i + 1:]:
            if b.offset < c.offset + c.nbytes and c.offset < b.offset + b.nbytes:
                assert live[b.id][1] < live[c.id][0] or live[c.id][1] < live[b.id][0], (b, c)
    for k, s in enumerate(plan.steps):
        for t in plan.steps[k + 1:]:
            if "group" in s.attrs and s.attrs["group"] == t.attrs.get("group"):
                assert set(s.writes).isdisjoint(t.reads + t.writes) and set(s.reads).isdisjoint(t.writes)
    monkeypatch.setattr(Planner, "_group_products", lambda self: None)
    alone, want = layers(dtype, optimizer)
    assert sorted(s.kind for s in alone.steps) == sorted(s.kind for s in plan.steps)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
