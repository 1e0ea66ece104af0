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
