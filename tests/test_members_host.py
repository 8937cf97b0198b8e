"""Products of one matrix that join one launch: which do, and that their results are theirs (on the numpy interpreter
of the launch records)."""
import numpy as np
import pytest

import nabla_amd as nb
from nabla_amd.core import engine


def planned(f, *args):
    engine.clear_plan_cache()
    out = f(*args)
    nb.realize_all(*out)
    steps = [s for bp in engine._PLAN_CACHE.values() for s in bp.plan.steps]
    engine.clear_plan_cache()
    return [o.numpy() for o in out], [s for s in steps if s.kind == "gemm"]


def tensors(*shapes):
    rng = np.random.default_rng(3)
    return [nb.Tensor.constant(rng.integers(-3, 4, s).astype(np.float32)) for s in shapes]


def test_projections_join_and_keep_their_own_biases(emulator):
    x, w1, w2, w3, b1, b3 = tensors((160, 64), (64, 96), (64, 96), (64, 96), (1, 96), (1, 96))

    def f(x, w1, w2, w3, b1, b3):
        return x @ w1 + b1, x @ w2, x @ w3 + b3

    on, steps = planned(f, x, w1, w2, w3, b1, b3)
    assert len(steps) == 1 and len(steps[0].attrs["members"]) == 3
    X, W1, W2, W3, B1, B3 = (t.numpy() for t in (x, w1, w2, w3, b1, b3))
    for got, want in zip(on, (X @ W1 + B1, X @ W2, X @ W3 + B3)):
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("case", ["width", "orientation", "depends", "rows"])
def test_others_stay_alone(emulator, case):
    x, w, v, u = tensors((160, 64), (64, 96), (64, 96) if case != "width" else (64, 80),
                         (96, 64) if case == "orientation" else (160, 64))
    if case == "rows":  # (up to 128 rows)
        x = tensors((128, 64))[0]

    def f(x, w, v, u):
        if case == "orientation":
            return x @ w, x @ nb.swap_axes(u, 0, 1)
        if case == "depends":  # (the second weight is made of the first result)
            y = x @ w
            return y, x @ (nb.swap_axes(x, 0, 1) @ y)
        return x @ w, x @ v

    got, steps = planned(f, x, w, v, u)
    assert not any(s.attrs.get("members") for s in steps)
    X, W, V, U = (t.numpy() for t in (x, w, v, u))
    want = (X @ U.T) if case == "orientation" else X @ (X.T @ (X @ W)) if case == "depends" else X @ V
    np.testing.assert_allclose(got[0], X @ W)
    np.testing.assert_allclose(got[1], want)
