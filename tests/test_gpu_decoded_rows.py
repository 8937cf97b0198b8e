"""Row programs whose inputs are read again in a later phase, with more values alive than the
interpreter's registers hold: results are comparisons and selections, exact in float32."""
import numpy as np
import pytest
import torch

import nabla_amd as nb
from nabla_amd.core import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_inputs", [6, 8, 9])
@pytest.mark.parametrize("cols", [5, 130, 1003, 4099])
def test_inputs_selected_again_after_a_reduction(hip, n_inputs, cols):
    rng = np.random.default_rng(n_inputs)
    xs = [rng.integers(-9, 10, (33, cols)).astype(np.float32) for _ in range(n_inputs)]

    def f(where, greater, reduce_max, xs):
        v = [greater(xs[k], xs[k - 1]) for k in range(n_inputs)]  # (x0 against the last)
        t = xs[0]
        for k in range(n_inputs):
            t = where(v[k], xs[k], t)
        o = reduce_max(t)
        for k in range(n_inputs):
            o = where(v[k], o, xs[k])
        return o

    engine.clear_plan_cache()
    hip.force_interpreter = True
    try:
        got = f(nb.where, nb.greater, lambda t: nb.reduce_max(t, axis=1, keepdims=True),
                [nb.Tensor.constant(x) for x in xs]).to_torch().cpu()
    finally:
        hip.force_interpreter = False
        engine.clear_plan_cache()
    want = f(torch.where, torch.gt, lambda t: t.max(1, keepdim=True).values, [torch.tensor(x) for x in xs])
    assert torch.equal(got, want)
