"""The decoder's last two layers in one kernel (sfh_nn_conv_t_out) against the
two separate ones, at image sizes around its tiles' edges, and a backward
after a prediction (which leaves out what the backward reads)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("B,Hi,Wi", [(1, 1, 1), (2, 4, 19), (1, 5, 20), (3, 8, 18), (2, 13, 38), (1, 52, 76)])
@pytest.mark.parametrize("dtype", [0, 1])
def test_equals_separate_layers(sfh, gpu_ctx, dtype, B, Hi, Wi, keep):
    import torch
    C, lib, h = 32, gpu_ctx.lib, gpu_ctx.handle
    g = torch.Generator(device="cuda").manual_seed(Hi * Wi + B)
    t = torch.bfloat16 if dtype == 0 else torch.float32
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    a, w = rnd(B, Hi, Wi, C).to(t), (0.1 * rnd(16 * C, C)).to(t)
    bias, w1, bmap = rnd(C), 0.2 * rnd(16, C), rnd(16 * Hi * Wi)
    pre, pre2 = torch.empty(B * 4 * Hi * Wi * C, device="cuda"), torch.full((B * 4 * Hi * Wi * C,), 7.0, device="cuda")
    out, out2 = torch.empty(B * 16 * Hi * Wi, device="cuda"), torch.empty(B * 16 * Hi * Wi, device="cuda")
    torch.cuda.synchronize()
    gpu_ctx.check(lib.sfh_nn_conv_t_fwd(h, dtype, a.data_ptr(), B, Hi, Wi, C, w.data_ptr(), bias.data_ptr(),
                                        pre.data_ptr(), None))
    gpu_ctx.check(lib.sfh_nn_conv1_fwd(h, pre.data_ptr(), B, 2 * Hi, 2 * Wi, C, w1.data_ptr(), bmap.data_ptr(), 1,
                                       out.data_ptr()))
    gpu_ctx.check(lib.sfh_nn_conv_t_out(h, dtype, a.data_ptr(), B, Hi, Wi, C, w.data_ptr(), bias.data_ptr(),
                                        w1.data_ptr(), bmap.data_ptr(), pre2.data_ptr() if keep else None,
                                        out2.data_ptr()))
    gpu_ctx.synchronize()
    # FP32 sums of 128 products of size ~0.1 and of 128 of size ~0.2, in another
    # order: 128 roundings of the partial sums (|sum| < 10) at most
    tol = 128 * 2.0 ** -24 * 10
    assert float((out - out2).abs().max()) <= 2 * tol
    if keep:
        assert float((pre - pre2).abs().max()) <= tol
    else:
        assert float(pre2.min()) == float(pre2.max()) == 7.0


def test_activation_over_the_whole_range(sfh, gpu_ctx):
    """SiLU of pre-activations up to the largest FP32 number, infinities and NaN,
    as biases of layers without weights: sfh_nn_conv_t_act rounds them to BF16
    (2^-9), sfh_nn_conv_t_out sums them with FP32 weights (each output adds four
    taps' sums of 32 channels, one of them non-zero here)."""
    import torch
    C, lib, h, n = 32, gpu_ctx.lib, gpu_ctx.handle, 2 * 3
    v = torch.tensor([-3.4e38, -1e30, -1e10, -1e3, -120.0, -100.0, -90.0, -88.8, -88.0, -87.0, -80.0, -40.0, -17.0, -5.0,
                      -1.0, -1e-3, 0.0, 1e-20, 0.5, 3.0, 20.0, 90.0, 1e10, 3.3e38, float("inf"), float("nan"),
                      -2.0, 2.0, -7.0, 7.0, -60.0, 60.0], device="cuda")
    want = torch.where(v < -700.0, torch.zeros_like(v).double(), v.double() / (1.0 + torch.exp(-v.double())))
    a = torch.zeros(n * C, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(16 * C * C, dtype=torch.bfloat16, device="cuda")
    act = torch.empty(4 * n, C, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    gpu_ctx.check(lib.sfh_nn_conv_t_act(h, 0, a.data_ptr(), 1, 2, 3, C, w.data_ptr(), v.data_ptr(), act.data_ptr()))
    gpu_ctx.synchronize()
    out = torch.empty(16 * n, device="cuda")
    for c in range(C):
        ok = torch.isfinite(want[c])
        got = act[:, c].double()
        if bool(ok):
            assert float((got - want[c]).abs().max()) <= 2.0 ** -8 * abs(float(want[c])) + 2e-36, float(v[c])
        else:
            assert bool((got.isnan() if v[c].isnan() else got == want[c]).all()), float(v[c])
        # exp's argument x log2 e is rounded: |x| 2^-24 of exp(-x), which matters
        # for x < 0 above -100; the reciprocal, the sums and products 2^-20
        rel = 2.0 ** -20 + min(abs(float(v[c])), 100.0) * 2.0 ** -24
        # one channel alone
        bias, w1 = torch.zeros(C, device="cuda"), torch.zeros(16, C, device="cuda")
        bias[c], w1[:, c] = v[c], 0.125
        torch.cuda.synchronize()
        gpu_ctx.check(lib.sfh_nn_conv_t_out(h, 0, a.data_ptr(), 1, 2, 3, C, w.data_ptr(), bias.data_ptr(),
                                            w1.data_ptr(), None, None, out.data_ptr()))
        gpu_ctx.synchronize()
        got = out.view(8, 12)[1:-1, 1:-1].double()
        if bool(ok):
            assert float((got - 0.5 * want[c]).abs().max()) <= rel * abs(float(want[c])) + 1e-36, float(v[c])
        else:
            assert bool((~got.isfinite()).all()), float(v[c])


def test_backward_after_prediction(sfh, gpu_ctx):
    import torch
    from sfh_amd import surrogate as S
    P = S.sample_parameters(3, seed=1)
    target = torch.randn((3, S.CROP_H, S.CROP_W), generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
    net = S.TemplateSurrogate(dtype="bf16", seed=3, max_batch=3)
    net.forward(P)
    loss = net.backward(target)
    g = net.gradient()
    net.forward(P[::-1])
    net.predict(P)
    assert net.backward(target) == loss
    assert np.array_equal(net.gradient(), g)
