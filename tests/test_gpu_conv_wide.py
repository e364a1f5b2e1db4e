"""The 8-wave convolution tiles against FP64 sums of the same BF16 values:
both tile shapes, both epilogues, the first sizes that take them and the last
that do not."""
import numpy as np
import pytest
import torch

from symphas_amd import nn

pytestmark = pytest.mark.gpu


# (N, H, W, C, K): 128 workgroups and more take the wide tiles (K % 128 == 0
# and H % 16 == 0, or K % 64 == 0 and H % 32 == 0); 127 do not
@pytest.mark.parametrize("act", [nn.ACT_NONE, nn.ACT_SILU])
@pytest.mark.parametrize("epi", [nn.EPI_PLAIN, nn.EPI_UPADD])
@pytest.mark.parametrize("N,H,W,C,K", [
    (64, 16, 32, 64, 128), (32, 32, 16, 96, 256), (128, 16, 16, 64, 384),
    (127, 16, 16, 64, 128), (64, 32, 32, 64, 64), (43, 32, 48, 96, 192),
    (127, 32, 16, 64, 64), (128, 16, 16, 64, 64), (128, 32, 16, 32, 64)])
def test_wide_tiles(gpu_lib, N, H, W, C, K, epi, act):
    print("[case] wide conv", N, H, W, C, K, epi, act, flush=True)
    g = torch.Generator(device="cuda").manual_seed(H * 100 + C)
    x = torch.randn(N, H, W, C, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(9, K, C, device="cuda", generator=g) / np.sqrt(9 * C)).to(torch.bfloat16)
    b = torch.randn(K, device="cuda", generator=g)
    skip = None
    if epi == nn.EPI_UPADD:
        skip = torch.randn(N, 2 * H, 2 * W, K, device="cuda", generator=g).to(torch.bfloat16)
    y, pre = nn.conv3x3_raw(x, w, b, act, epi, skip, want_pre=True)
    want = b.double().expand(N * H * W, K).clone()
    for t in range(9):
        v = torch.roll(x, (1 - t // 3, 1 - t % 3), dims=(1, 2)).reshape(-1, C).double()
        want += v @ w[t].double().t()
    want = want.view(N, H, W, K)
    if epi == nn.EPI_UPADD:
        want = want.repeat_interleave(2, 1).repeat_interleave(2, 2) + skip.double()
    # one BF16 rounding of an FP32 sum: half an ulp of the value and the
    # rounding of 9*C products of unit variance in FP32
    tol = want.abs() * 2.0 ** -8 + 9 * C * 2.0 ** -22
    assert bool(((pre.double() - want).abs() <= tol).all())
    if act == nn.ACT_SILU:
        want = want * torch.sigmoid(want)
        tol = want.abs() * 2.0 ** -8 + 9 * C * 2.0 ** -21
    assert bool(((y.double() - want).abs() <= tol).all())
    y2, _ = nn.conv3x3_raw(x, w, b, act, epi, skip)
    assert torch.equal(y, y2)
