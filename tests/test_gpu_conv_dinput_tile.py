"""The decoder's input gradient from tiles (BF16, 32 channels) where tiles of
6 x 19 pixels end: against the FP64 product of the same rounded operands, and
a strided output that the tile form leaves to the gathering form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hi,Wi", [(1, 1, 1), (2, 5, 18), (3, 6, 19), (1, 7, 20), (2, 12, 38), (1, 13, 39)])
@pytest.mark.parametrize("ldo", [32, 36, 33])
def test_conv_dinput_tiles(sfh, gpu_ctx, B, Hi, Wi, ldo):
    import torch
    rng = np.random.default_rng(100 * Hi + Wi)
    C = 32
    d = torch.from_numpy(rng.normal(size=(B, 2 * Hi, 2 * Wi, C)).astype(np.float32)).cuda()
    wT = torch.from_numpy(rng.normal(size=(C, 16 * C)).astype(np.float32)).cuda().to(torch.bfloat16)
    out = torch.full((B * Hi * Wi, ldo), -7.0, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    gpu_ctx.check(gpu_ctx.lib.sfh_nn_conv_t_dinput(gpu_ctx.handle, 0, d.data_ptr(), B, Hi, Wi, C, wT.data_ptr(),
                                                   16 * C, C, out.data_ptr(), ldo))
    gpu_ctx.synchronize()
    dp = np.zeros((B, 2 * Hi + 2, 2 * Wi + 2, C))
    dp[:, 1:-1, 1:-1] = d.to(torch.bfloat16).double().cpu().numpy()
    w = wT.double().cpu().numpy().reshape(C, 4, 4, C)
    ref, mag = np.zeros((B, Hi, Wi, C)), np.zeros((B, Hi, Wi, C))
    for ky in range(4):
        for kx in range(4):
            v = dp[:, ky:ky + 2 * Hi:2, kx:kx + 2 * Wi:2]
            ref += v @ w[:, ky, kx].T
            mag += np.abs(v) @ np.abs(w[:, ky, kx].T)
    got = out.cpu().numpy().astype(np.float64)
    # 512 exact products added in FP32: at most 512 roundings of 2^-24 of the sum of magnitudes
    assert np.all(np.abs(got[:, :C].reshape(ref.shape) - ref) <= 512 * 2.0 ** -24 * mag)
    assert np.all(got[:, C:] == -7.0)
