"""The row-program interpreter at the edges of its launch forms: rows shared by a wavefront
(up to 32 chunks of 4 columns), rows of one and several wavefronts, the longest row held in
registers (1024 chunks), longer rows, rows whose start no vector access is aligned to, and inputs
it can and cannot request ahead."""
import numpy as np
import pytest
import torch

import nabla_amd as nb

pytestmark = pytest.mark.gpu


@pytest.fixture
def interpreted(hip):
    from nabla_amd.core import engine
    engine.clear_plan_cache()
    hip.force_interpreter = True
    yield hip
    hip.force_interpreter = False
    engine.clear_plan_cache()


def tensor(a, dtype):
    return nb.Tensor.from_dlpack(torch.tensor(a).to(getattr(torch, dtype)).cuda())


def stored(t):
    return t.to_torch().double().cpu()


# One row program of three phases: five rounded operations per element at most lie between an
# input and a result of order one, sums of C terms add log2(C) more in a tree; 2e-6 relative
# of the row's largest value covers both at fp32.  A bf16 result is rounded once: 2^-9.
@pytest.mark.parametrize("cols", [1, 3, 4, 5, 8, 31, 64, 86, 127, 128, 129, 255, 257, 1003, 2048, 2051, 4096, 4099, 9001])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_rows_of_every_length(interpreted, cols, dtype):
    rows = 77
    rng = np.random.default_rng(cols)
    x, g, t = (tensor(rng.standard_normal((rows, cols)).astype(np.float32), dtype) for _ in range(3))
    keep = nb.Tensor.constant(rng.random((rows, cols)) < 0.7)
    w = tensor(rng.standard_normal(cols).astype(np.float32), dtype)

    def f(x, g):
        z = nb.where(keep, x * nb.sigmoid(g) + w, x - t)
        m = nb.reduce_max(z, axis=1, keepdims=True)
        e = nb.exp(z - m)
        return e / nb.reduce_sum(e, axis=1, keepdims=True), m

    p, m = f(x, g)
    nb.realize_all(p, m)
    X, G, W, U = stored(x), stored(g), stored(w), stored(t)
    z = torch.where(torch.tensor(keep.numpy()), X * torch.sigmoid(G) + W, X - U)
    want = torch.softmax(z, 1)
    tol = 4e-6 if dtype == "float32" else 2.0 ** -8
    assert ((stored(p) - want).abs() <= tol * want.abs() * (1 + z.abs().max())).all()
    assert ((stored(m)[:, 0] - z.max(1).values).abs() <= tol * (1 + z.abs().max())).all()


@pytest.mark.parametrize("n_inputs", [1, 6, 9, 12])
def test_many_inputs_shared_by_two_phases(interpreted, n_inputs):
    """More inputs than are requested ahead, each read before and after a reduction."""
    rows, cols = 130, 200
    rng = np.random.default_rng(n_inputs)
    xs = [tensor(rng.standard_normal((rows, cols)).astype(np.float32), "float32") for _ in range(n_inputs)]
    total = xs[0] * 0.5
    for k, x in enumerate(xs[1:]):
        total = total + x * nb.exp(x * (0.1 * (k + 1)))
    s = nb.reduce_sum(total, axis=1, keepdims=True)
    out = total * s
    for x in xs:
        out = out + x * s
    nb.realize_all(out, s)
    X = [stored(x) for x in xs]
    want = X[0] * 0.5
    for k, x in enumerate(X[1:]):
        want = want + x * torch.exp(x * (0.1 * (k + 1)))
    mag = want.abs().sum(1, keepdim=True)
    ws = want.sum(1, keepdim=True)
    assert ((stored(s) - ws).abs() <= 2e-6 * mag).all()
    wo = want * ws + sum(x * ws for x in X)
    bound = 2e-6 * (want.abs() * mag + sum(x.abs() * mag for x in X) + wo.abs())
    assert ((stored(out) - wo).abs() <= bound).all()


@pytest.mark.parametrize("shape", [(3, 5, 7), (64, 1, 33), (2, 300, 130), (1, 1, 2049)])
def test_elementwise_over_broadcast_and_transposed_operands(interpreted, shape):
    b, r, c = shape
    rng = np.random.default_rng(r)
    x = tensor(rng.standard_normal((b, r, c)).astype(np.float32), "float32")
    y = tensor(rng.standard_normal((b, c, r)).astype(np.float32), "float32")
    row = tensor(rng.standard_normal((b, r, 1)).astype(np.float32), "float32")
    col = tensor(rng.standard_normal((1, 1, c)).astype(np.float32), "bfloat16")
    n = nb.Tensor.constant(rng.integers(-9, 9, (b, r, c)).astype(np.int32))
    out = nb.tanh(x + nb.swap_axes(y, 1, 2) * row) + nb.cast(col, nb.DType.float32) * nb.cast(n, nb.DType.float32)
    big = nb.greater(out, 0.0)
    nb.realize_all(out, big)
    want = torch.tanh(stored(x) + stored(y).transpose(1, 2) * stored(row)) + stored(col) * stored(n)
    assert ((stored(out) - want).abs() <= 2e-6 * (1 + want.abs())).all()
    sure = want.abs() > 1e-4
    assert (torch.tensor(big.numpy())[sure] == (want > 0)[sure]).all()


@pytest.mark.parametrize("cols", [255, 256, 257, 262, 511, 512, 513, 519, 2046, 4095, 4096])
@pytest.mark.parametrize("live", [3, 12])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_one_and_two_chunks_a_lane(interpreted, cols, live, dtype):
    """Up to 64 chunks a lane holds one, from there on two if the program has at most eight vectors alive at a
    time.  Whole numbers below 256: exact in both types."""
    rows = 70
    rng = np.random.default_rng(cols + live)
    xs = [rng.integers(-3, 4, (rows, cols)).astype(np.float32) for _ in range(live)]

    def f(*xs):
        total = xs[0]
        for i, x in enumerate(xs[1:]):
            total = total + x if i % 2 else total - x
        top = nb.reduce_max(total, axis=1, keepdims=True)
        low = nb.reduce_min(total, axis=1, keepdims=True)
        out = top - total
        for x in xs:
            out = out + (x - nb.relu(x)) * nb.where(x > low, x, low * 0.0)
        return out, top, low

    got = f(*(tensor(x, dtype) for x in xs))
    nb.realize_all(*got)
    total = xs[0].copy()
    for i, x in enumerate(xs[1:]):
        total = total + x if i % 2 else total - x
    top, low = total.max(1, keepdims=True), total.min(1, keepdims=True)
    out = top - total
    for x in xs:
        out = out + np.minimum(x, 0) * np.where(x > low, x, 0)
    assert np.abs(out).max() < 256
    for g, w in zip(got, (out, top, low)):
        np.testing.assert_array_equal(stored(g).numpy(), w)
