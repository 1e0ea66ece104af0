"""The output layer's input and weight gradients from one pass, where blocks of
16 pixels cross rows and images: the input gradient is that of a call without
the weight gradient to the bit, and the weight gradient that of a call of its
own up to the order of its FP32 sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("B,H,W", [(1, 1, 1), (2, 1, 3), (3, 5, 1), (2, 7, 16), (5, 9, 11), (40, 52, 38)])
def test_conv1_bwd_one_pass(sfh, gpu_ctx, B, H, W, act):
    import torch
    rng = np.random.default_rng(1000 * B + 10 * H + W)
    C, P = 32, B * H * W
    def dev(shape):
        return torch.from_numpy(rng.normal(size=shape).astype(np.float32)).cuda()
    dout, x, w = dev((B, 2 * H, 2 * W)), dev((P, C)), dev((16, C))
    din, dw = [torch.full_like(x, float("nan")) for _ in range(2)], [torch.full_like(w, float("nan")) for _ in range(2)]
    dsum = [torch.full((C,), float("nan"), device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    def call(di, ds, dk):
        gpu_ctx.check(gpu_ctx.lib.sfh_nn_conv1_bwd(gpu_ctx.handle, dout.data_ptr(), x.data_ptr(), B, H, W, C,
                                                   w.data_ptr(), act, di, ds, dk, None))
    call(din[0].data_ptr(), dsum[0].data_ptr(), dw[0].data_ptr())
    call(din[1].data_ptr(), dsum[1].data_ptr(), None)
    call(None, None, dw[1].data_ptr())
    gpu_ctx.synchronize()
    assert torch.equal(din[0], din[1])
    x64 = x.double()
    a = x64 * torch.sigmoid(x64) if act else x64
    pad = torch.nn.functional.pad(dout.double(), (1, 1, 1, 1))
    win = torch.stack([pad[:, ky:ky + 2 * H:2, kx:kx + 2 * W:2].reshape(P) for ky in range(4) for kx in range(4)])
    # sums of P FP32 products: 2^-24 per operation of the running magnitude, which the split over at
    # most 1024 workgroups and 4 waves bounds by P / 1024 + 1040 operations; 2^-20 for the activation
    ref, mag = win @ a, win.abs() @ a.abs()
    tol = ((P / 1024 + 1040) * 2.0 ** -24 + 2.0 ** -20) * mag
    for d in dw:
        assert torch.all((d.double() - ref).abs() <= tol)
    d64 = din[0].double()
    for s in dsum:
        assert torch.all((s.double() - d64.sum(0)).abs() <= (P / 1024 + 2100) * 2.0 ** -24 * d64.abs().sum(0))
