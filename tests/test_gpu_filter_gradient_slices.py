"""Filter gradients as sums of slices of the contraction: few slices and many, by sixteen, by four and by one lane
a sum, results that leave a workgroup's last columns empty.  Whole numbers, whose sums are exact."""
import numpy as np
import pytest
import torch

import nabla_amd as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hw,cin,cout", [
    (2, 12, 3, 5), (7, 13, 7, 9), (20, 16, 3, 17), (70, 22, 1, 24), (64, 32, 3, 64),  # sixteen lanes: 4 to 512 slices
    (3, 20, 40, 45), (9, 11, 40, 72), (31, 17, 64, 56), (16, 24, 64, 96),              # four
    (6, 10, 130, 120), (5, 19, 128, 136)])                                             # one
def test_slices_add_up(hip, n, hw, cin, cout):
    rng = np.random.default_rng(cout)
    x = rng.integers(-4, 5, (n, hw, hw, cin)).astype(np.float32)
    w = rng.integers(-4, 5, (3, 3, cin, cout)).astype(np.float32)
    g = rng.integers(-4, 5, (n, hw, hw, cout)).astype(np.float32)
    T = nb.Tensor.constant
    got = nb.grad(lambda b: nb.reduce_sum(nb.conv2d(T(x), b, padding=(1, 1, 1, 1)) * T(g)))(T(w)).numpy()
    image = torch.nn.functional.pad(torch.tensor(x, dtype=torch.float64), (0, 0, 1, 1, 1, 1))
    dy = torch.tensor(g, dtype=torch.float64).reshape(-1, cout)
    want = np.stack([[(image[:, r:r + hw, s:s + hw].reshape(-1, cin).T @ dy).numpy() for s in range(3)] for r in range(3)])
    np.testing.assert_array_equal(got, want)
