"""Forward convolutions with up to 32 numbers a channel of the result: 1 to 16 steps, columns at the edges of the blocks
of 32, fewer pixels than a block and more than the launch has waves for, strides, relu.  Whole numbers, whose sums are exact."""
import numpy as np
import pytest

import nabla_amd as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,cin,cout,r,s,pad,stride", [
    (1, 1, 1, 1, 1, 1, 1, 0, 1), (1, 2, 3, 3, 31, 3, 3, 1, 1), (5, 40, 1, 3, 33, 3, 1, 0, 1), (3, 1, 37, 2, 32, 1, 3, 0, 1),
    (9, 13, 11, 1, 65, 5, 5, 2, 1), (7, 17, 14, 3, 64, 3, 3, 1, 2), (6, 19, 23, 32, 40, 1, 1, 0, 1), (150, 31, 32, 17, 24, 1, 1, 0, 1),
    (11, 30, 29, 8, 130, 2, 2, 0, 3), (4, 9, 9, 16, 16, 1, 1, 1, 1)])
@pytest.mark.parametrize("relu", [False, True])
def test_few_numbers(hip, n, h, w, cin, cout, r, s, pad, stride, relu):
    rng = np.random.default_rng(n)
    ho, wo = (h + 2 * pad - r) // stride + 1, (w + 2 * pad - s) // stride + 1
    x = rng.integers(-4, 5, (n, h, w, cin)).astype(np.float32)
    k = rng.integers(-4, 5, (r, s, cin, cout)).astype(np.float32)
    bias = rng.integers(-4, 5, (cout,)).astype(np.float32)
    T = nb.Tensor.constant
    y = nb.conv2d(T(x), T(k), stride=(stride, stride), padding=(pad,) * 4, bias=T(bias))
    got = (nb.relu(y) if relu else y).numpy()
    image = np.pad(x, ((0, 0), (pad, pad), (pad, pad), (0, 0)))
    want = sum(image[:, a:a + stride * (ho - 1) + 1:stride, b:b + stride * (wo - 1) + 1:stride].reshape(-1, cin) @ k[a, b]
               for a in range(r) for b in range(s)).reshape(n, ho, wo, cout) + bias
    np.testing.assert_array_equal(got, np.maximum(want, 0) if relu else want)
