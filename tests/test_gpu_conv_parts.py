"""Convolutions out of bf16 parts: forward, input and filter gradient at the edges of their tiles (128 x 128,
64 x 64, 128 x 32) and of a K tile, in pieces of eight channels and number by number, against float64;
numbers that have no parts."""
import numpy as np
import pytest
import torch

import nabla_amd as nb

pytestmark = pytest.mark.gpu


def ours(x, w, g, pad, stride):
    def loss(a, b):
        return nb.reduce_sum(nb.conv2d(a, b, stride=(stride, stride), padding=(pad,) * 4) * T(g))
    T = nb.Tensor.constant
    y = nb.conv2d(T(x), T(w), stride=(stride, stride), padding=(pad,) * 4).numpy()
    return [y] + [t.numpy() for t in nb.grad(loss, argnums=(0, 1))(T(x), T(w))]


def reference(x, w, g, pad, stride):
    """The three results in float64."""
    tx = torch.tensor(x, dtype=torch.float64).permute(0, 3, 1, 2).requires_grad_()
    tw = torch.tensor(w, dtype=torch.float64).permute(3, 2, 0, 1).requires_grad_()
    y = torch.nn.functional.conv2d(tx, tw, padding=pad, stride=stride)
    dx, dw = torch.autograd.grad(y, (tx, tw), torch.tensor(g, dtype=torch.float64).permute(0, 3, 1, 2))
    return [y.detach().permute(0, 2, 3, 1).numpy(), dx.permute(0, 2, 3, 1).numpy(), dw.permute(2, 3, 1, 0).numpy()]


@pytest.mark.parametrize("n,hw,cin,cout,r,pad,stride", [
    (33, 32, 8, 32, 3, 1, 1), (37, 31, 5, 31, 3, 1, 1),      # results of up to 32 channels: 128 x 32
    (32, 33, 64, 130, 3, 1, 1), (41, 29, 20, 128, 3, 0, 1),  # 128 x 128
    (2, 9, 24, 65, 3, 1, 2), (3, 8, 7, 64, 1, 0, 1),         # 64 x 64, a K tile and less
    (1, 5, 1, 1, 3, 1, 1), (3, 12, 16, 40, 5, 2, 1)])
def test_against_float64(hip, n, hw, cin, cout, r, pad, stride):
    rng = np.random.default_rng(cin)
    ho = (hw + 2 * pad - r) // stride + 1
    x = rng.standard_normal((n, hw, hw, cin)).astype(np.float32)
    w = rng.standard_normal((r, r, cin, cout)).astype(np.float32)
    g = rng.standard_normal((n, ho, ho, cout)).astype(np.float32)
    got = ours(x, w, g, pad, stride)
    want = reference(x, w, g, pad, stride)
    size = reference(np.abs(x), np.abs(w), np.abs(g), pad, stride)
    # a sum is rounded once per K tile of 32 and accumulator (2^-24 of the sum of magnitudes at most) and once in
    # each small product; the filter gradient on the float32 instruction once per two numbers
    # of a slice of K, in the worst case
    for a, c, s, terms in zip(got, want, size, (r * r * cin / 32, r * r * cout / 32, n * ho * ho / 2)):
        assert (np.abs(a - c) <= (terms + 6) * 2.0 ** -24 * s + 2.0 ** -23 * np.abs(c)).all()


@pytest.mark.parametrize("n,hw", [(3, 7), (130, 16)])
@pytest.mark.parametrize("cin,cout,r", [(33, 64, 1), (64, 33, 1), (65, 96, 1), (97, 72, 1), (128, 100, 1), (100, 128, 1),
                                        (129, 136, 1), (136, 129, 1), (3, 37, 5), (11, 12, 3), (14, 15, 3)])
def test_contractions_of_one_to_five_tiles(hip, n, hw, cin, cout, r):
    """Those of up to four K tiles request no more than they have; filter gradients in short slices, too."""
    rng = np.random.default_rng(cin)
    x, g = (rng.standard_normal((n, hw, hw, c)).astype(np.float32) for c in (cin, cout))
    w = rng.standard_normal((r, r, cin, cout)).astype(np.float32)
    a, b = (r // 2, 1), (np.abs(x), np.abs(w), np.abs(g))
    for got, want, size, terms in zip(ours(x, w, g, *a), reference(x, w, g, *a), reference(*b, *a),
                                      (r * r * cin / 32, r * r * cout / 32, n * hw * hw / 2)):
        assert (np.abs(got - want) <= (terms + 6) * 2.0 ** -24 * size + 2.0 ** -23 * np.abs(want)).all()


@pytest.mark.parametrize("n,hw,cin", [(33, 32, 8), (32, 32, 128), (2, 9, 65)])
def test_a_result_of_one_product_is_rounded_once(hip, n, hw, cin):
    """Input gradients of one output channel and one tap; filter gradients of one pixel."""
    rng = np.random.default_rng(cin)
    x, g = (rng.standard_normal((n, hw, hw, c)).astype(np.float32) for c in (cin, 1))
    w = rng.standard_normal((1, 1, cin, 1)).astype(np.float32)
    np.testing.assert_array_equal(ours(x, w, g, 0, 1)[1], g * w[0, 0, :, 0])
    x, w, g = (rng.standard_normal(s).astype(np.float32) for s in ((1, 1, 1, cin), (1, 1, cin, 37), (1, 1, 1, 37)))
    np.testing.assert_array_equal(ours(x, w, g, 0, 1)[2][0, 0], x[0, 0, 0][:, None] * g[0, 0, 0])


@pytest.mark.parametrize("n,hw,cin,cout", [(33, 32, 8, 32), (32, 32, 8, 128), (2, 9, 7, 65)])
def test_small_numbers(hip, n, hw, cin, cout):
    """Images and cotangents of a few digits of the smallest float32 kind, filters as much larger."""
    rng = np.random.default_rng(0)
    x, w, g = (np.ldexp(rng.standard_normal(s), e).astype(np.float32) for s, e in (
        ((n, hw, hw, cin), -130), ((3, 3, cin, cout), 70), ((n, hw, hw, cout), -120)))
    for a, c, s in list(zip(ours(x, w, g, 1, 1), reference(x, w, g, 1, 1),
                            reference(np.abs(x), np.abs(w), np.abs(g), 1, 1)))[:2]:
        assert (np.abs(a - c) <= (9 * max(cin, cout) / 32 + 6) * 2.0 ** -24 * s + 2.0 ** -23 * np.abs(c)).all()


@pytest.mark.parametrize("n,hw,cin,cout", [(33, 32, 8, 32), (32, 32, 8, 128), (2, 9, 7, 65)])
def test_numbers_without_parts(hip, n, hw, cin, cout):
    rng = np.random.default_rng(0)
    x = rng.uniform(0.5, 1.0, (n, hw, hw, cin)).astype(np.float32)
    w = rng.uniform(0.5, 1.0, (3, 3, cin, cout)).astype(np.float32)
    x[0, 1, 1, 0], x[n - 1, 4, 7, 3], x[0, 5, 5, 1] = np.inf, np.nan, 3.4e38  # (the last: infinity as a bf16)
    w[0, 0, 0, 3], w[1, 1, 1, 2] = 0.0, 1e-30                                # (infinity times zero)
    got = nb.conv2d(nb.Tensor.constant(x), nb.Tensor.constant(w), padding=(1, 1, 1, 1)).numpy()
    want = torch.nn.functional.conv2d(torch.tensor(x).double().permute(0, 3, 1, 2),
                                      torch.tensor(w).double().permute(3, 2, 0, 1), padding=1)
    want = want.permute(0, 2, 3, 1).numpy()
    over = np.abs(want) > 3.5e38
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    assert np.isinf(got[over]).all()
    ok = np.abs(want) < 3.3e38
    assert (np.abs(got[ok] - want[ok]) <= 1e-5 * np.abs(want[ok])).all()


def descriptor(n, hw, cin, cout, r):
    from nabla_amd.backend import lib
    d = lib.ConvDesc()
    d.N, d.H, d.W, d.Cin, d.R, d.S, d.Cout, d.Ho, d.Wo = n, hw, hw, cin, r, r, cout, hw, hw
    d.stride_h = d.stride_w = 1
    d.pad_t = d.pad_b = d.pad_l = d.pad_r = r // 2
    return d


def test_few_output_channels_cost_no_more_than_eight(hip):
    """Input gradients number by number, of one and two K tiles: with requests past the last tile those of four
    channels took 1.6 times as long as those of eight."""
    from nabla_amd.backend import lib
    from test_gpu_gemm_f32_parts import seconds
    st = lib.C.c_void_p(torch.cuda.current_stream().cuda_stream)
    times = []
    for cout in (8, 3, 4):
        d = descriptor(64, 32, 128, cout, 3)
        y, w, x = (torch.ones(s, device="cuda") for s in ((64, 32, 32, cout), (3, 3, 128, cout), (64, 32, 32, 128)))
        times.append(min(seconds(lambda: lib.check(lib.load().nbk_conv2d_dgrad(
            lib.C.byref(d), *(lib.C.c_void_p(t.data_ptr()) for t in (y, w, x)), st))) for _ in range(3)))
    assert max(times[1:]) <= 1.3 * times[0], times


@pytest.mark.parametrize("n,hw,cin,cout,r", [(81, 14, 140, 114, 3), (16, 28, 50, 50, 3), (64, 28, 30, 60, 3), (10, 30, 27, 237, 3)])
def test_slices_of_odd_filter_gradients_are_one_round(hip, n, hw, cin, cout, r):
    from nabla_amd.backend import lib
    d = descriptor(n, hw, cin, cout, r)
    rows = r * r * cin
    slices = lib.load().nbk_conv2d_wgrad_workspace(lib.C.byref(d)) // (4 * rows * cout)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert 1 < slices and slices * -(-rows // 64) * -(-cout // 64) <= 3 * cus


@pytest.mark.parametrize("cin,cout", [(64, 128), (20, 40)])
def test_numbers_without_parts_cost_one_more_pass(hip, cin, cout):
    """Images of NaN throughout: every wave runs its tile again on the float32 instruction and gathers number by
    number (one result after the other took 43 to 130 times as long)."""
    from nabla_amd.backend import lib
    from test_gpu_gemm_f32_parts import seconds
    d = lib.ConvDesc()
    d.N, d.H, d.W, d.Cin, d.R, d.S, d.Cout, d.Ho, d.Wo = 32, 32, 32, cin, 3, 3, cout, 32, 32
    d.stride_h = d.stride_w = d.pad_t = d.pad_b = d.pad_l = d.pad_r = 1
    w = torch.ones((3, 3, cin, cout), device="cuda")
    st = lib.C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: lib.C.c_void_p(t.data_ptr())
    L = lib.load()
    for run, ci, co in ((lambda x, y: L.nbk_conv2d_fwd(lib.C.byref(d), ptr(x), ptr(w), None, ptr(y), st), cin, cout),
                        (lambda x, y: L.nbk_conv2d_dgrad(lib.C.byref(d), ptr(x), ptr(w), ptr(y), st), cout, cin)):
        times = []
        for value in (1.0, float("nan")):
            x, y = torch.full((32, 32, 32, ci), value, device="cuda"), torch.empty((32, 32, 32, co), device="cuda")
            times.append(seconds(lambda: lib.check(run(x, y))))
            assert torch.isnan(y).all() == (value != value)
        assert times[1] <= 10 * times[0]
