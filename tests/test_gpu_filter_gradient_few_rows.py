"""Filter gradients of up to 32 filter rows: one row to 32, columns at the edges of the blocks of 32, fewer pixels than
half waves, images one pixel wide, strides, slices that are no multiple of the steps in flight.  Whole numbers,
whose sums are exact, and an infinity among them."""
import numpy as np
import pytest

import nabla_amd as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,cin,cout,r,s,pad,stride", [
    (1, 1, 1, 1, 1, 1, 1, 0, 1), (1, 2, 3, 3, 31, 3, 3, 1, 1), (5, 40, 1, 3, 33, 3, 1, 0, 1), (3, 1, 37, 2, 32, 1, 3, 0, 1),
    (9, 13, 11, 1, 65, 5, 5, 2, 1), (7, 17, 14, 3, 64, 3, 3, 1, 2), (6, 19, 23, 32, 40, 1, 1, 0, 1), (64, 32, 32, 3, 64, 3, 3, 1, 1),
    (11, 30, 29, 8, 130, 2, 2, 0, 3)])
@pytest.mark.parametrize("infinity", [False, True])
def test_few_rows(hip, n, h, w, cin, cout, r, s, pad, stride, infinity):
    rng = np.random.default_rng(n)
    ho, wo = (h + 2 * pad - r) // stride + 1, (w + 2 * pad - s) // stride + 1
    x = rng.integers(-4, 5, (n, h, w, cin)).astype(np.float32)
    k = rng.integers(-4, 5, (r, s, cin, cout)).astype(np.float32)
    g = rng.integers(-4, 5, (n, ho, wo, cout)).astype(np.float32)
    if infinity:
        x[n - 1, h - 1, w - 1, cin - 1] = np.inf
    T = nb.Tensor.constant
    got = nb.grad(lambda b: nb.reduce_sum(
        nb.conv2d(T(x), b, stride=(stride, stride), padding=(pad,) * 4) * T(g)))(T(k)).numpy()
    image = np.pad(x.astype(np.float64), ((0, 0), (pad, pad), (pad, pad), (0, 0)))
    with np.errstate(invalid="ignore"):
        want = np.stack([[np.einsum("nhwc,nhwj->cj",
                                    image[:, a:a + stride * (ho - 1) + 1:stride, b:b + stride * (wo - 1) + 1:stride],
                                    g.astype(np.float64), optimize=False) for b in range(s)] for a in range(r)])
    np.testing.assert_array_equal(got, want)
