"""Weight gradients x^T dy over a number of rows that no number of slices divides, as the planner cuts
them: whole numbers, every sum exact in float32, one rounding to bf16."""
import numpy as np
import pytest
import torch

import nabla_amd as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(512, 512, 8200), (512, 512, 9600), (256, 256, 8640), (2048, 16, 9216),
                                   (16, 16, 16400), (64, 24, 33000), (520, 264, 1100)])
def test_a_weight_gradient_over_many_rows(hip, M, N, K):
    rng = np.random.default_rng(K)
    x, g = rng.integers(-2, 3, (K, M)).astype(np.float32), rng.integers(-2, 3, (K, N)).astype(np.float32)
    xd, gd = (nb.Tensor.from_dlpack(torch.tensor(a).to(torch.bfloat16).cuda()) for a in (x, g))
    got = (nb.swap_axes(xd, 0, 1) @ gd).to_torch().double().cpu().numpy()
    want = x.T.astype(np.float64) @ g
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want)).all()
