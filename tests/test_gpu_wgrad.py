"""The tiled weight gradient and its bias gradient: chunk widths, part shapes,
remainders over workgroups, against FP64 sums of the same BF16 values."""
import numpy as np
import pytest
import torch

from symphas_amd import abi, nn

pytestmark = pytest.mark.gpu


# chunks of 32, 16 and 8 columns; 64 and 32 channel tiles; one chunk, more
# workgroups than chunks, a last workgroup with fewer; the general kernel
@pytest.mark.parametrize("N,H,W,C,K", [
    (1, 4, 32, 64, 64), (3, 8, 64, 64, 64), (2, 8, 16, 64, 64), (5, 16, 8, 64, 64),
    (1, 8, 32, 32, 32), (2, 16, 48, 32, 32), (1, 32, 24, 32, 32), (17, 24, 32, 32, 32),
    (1, 4, 32, 32, 64), (2, 8, 16, 32, 128), (1, 16, 40, 32, 64),
    (1, 4, 32, 64, 32), (2, 8, 48, 128, 32), (3, 16, 8, 64, 96),
    (2, 32, 32, 256, 128), (4, 64, 64, 64, 128), (1, 64, 320, 64, 64),
    (2, 4, 8, 64, 32), (1, 2, 32, 32, 64), (4, 3, 8, 32, 32)])
def test_weight_and_bias_gradients(gpu_lib, N, H, W, C, K):
    print("[case] wgrad", N, H, W, C, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(N * 1000 + W)
    x = torch.randn(N, H, W, C, device="cuda", generator=g).to(torch.bfloat16)
    d = torch.randn(N, H, W, K, device="cuda", generator=g).to(torch.bfloat16)
    dw, db = nn.conv3x3_wgrad_bias_raw(x, d, K)
    again = nn.conv3x3_wgrad_bias_raw(x, d, K)
    assert torch.equal(dw, again[0]) and torch.equal(db, again[1])
    assert torch.equal(dw, nn.conv3x3_wgrad_raw(x, d, K))
    xd, dd = x.double(), d.double().reshape(-1, K)
    # FP32 sums of npix products: rounding of a random walk, times a margin
    tol = 8 * 2.0 ** -24 * np.sqrt(N * H * W)
    for t in range(9):
        v = torch.roll(xd, (1 - t // 3, 1 - t % 3), dims=(1, 2)).reshape(-1, C)
        want = dd.t() @ v
        scale = float((dd.abs().t() @ v.abs()).max()) / np.sqrt(N * H * W)
        assert float((dw[t].double() - want).abs().max()) <= tol * scale, t
    scale = float(dd.abs().sum(0).max()) / np.sqrt(N * H * W)
    assert float((db.double() - dd.sum(0)).abs().max()) <= tol * scale


# tiled, general and thin kernels, with 256 to 2048 partial sums
@pytest.mark.parametrize("N,H,W,thin", [(32, 256, 256, False), (8, 100, 100, False),
                                        (32, 256, 256, True), (8, 100, 90, True)])
def test_bias_gradient_sums_keep_their_precision(gpu_lib, N, H, W, thin):
    # positive sums of up to 2 million values: a workgroup's own sum is off by a
    # few units of its last place, independent of the others', and their sum
    # adds its one rounding, at most 2^-24 of every value
    g = torch.Generator(device="cuda").manual_seed(H)
    d = (torch.randn(N, H, W, 32, device="cuda", generator=g) * 0.1 + 0.05).to(torch.bfloat16)
    if thin:
        out = torch.zeros(10, 32, device="cuda")
        s = torch.randn(N, H, W, device="cuda", generator=g)
        ws = nn.wgrad_workspace(nn.WGRAD_IN1, N, H, W, 1, 32, "cuda")
        nn._check(abi.load().sps_nn_conv3x3_in1_wgrad_bias(
            nn._ptr(s), nn._ptr(d), N, H, W, 32, nn._ptr(out), nn._ptr(out[9]), nn._ptr(ws),
            ws.numel(), nn._stream()))
        db = out[9]
    else:
        db = nn.conv3x3_wgrad_bias_raw(torch.zeros_like(d), d, 32)[1]
    want = d.double().sum((0, 1, 2))
    assert float((db.double() - want).norm() / want.norm()) <= 2.0 ** -24


@pytest.mark.parametrize("N,H,W,C,K", [(56, 24, 24, 256, 256), (8, 64, 64, 64, 64)])
def test_the_bias_gradient_costs_no_pass_of_its_own(gpu_lib, N, H, W, C, K):
    # general and tiled kernel: a product with ones beside nine of each tap's
    # (1/9 of the products at most), against twice the time with a serial pass
    x = torch.zeros(N, H, W, C, device="cuda", dtype=torch.bfloat16)
    d = torch.zeros(N, H, W, K, device="cuda", dtype=torch.bfloat16)

    def best(f):
        times = []
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(20):
                f(x, d, K)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert best(nn.conv3x3_wgrad_bias_raw) <= 1.5 * best(nn.conv3x3_wgrad_raw)


# one run of 64 pixels, a part of one, rows shorter than a run, several and
# more than 1024 workgroups' least; channels that leave waves idle
@pytest.mark.parametrize("N,H,W,C", [(1, 8, 8, 32), (1, 5, 7, 8), (3, 3, 3, 16), (2, 9, 70, 24),
                                     (1, 1, 2000, 64), (5, 128, 128, 32), (2, 200, 331, 40),
                                     (3, 700, 601, 8)])
def test_thin_gradients(gpu_lib, N, H, W, C):
    print("[case] thin wgrad", N, H, W, C, flush=True)
    lib = abi.load()
    g = torch.Generator(device="cuda").manual_seed(W)
    a = torch.randn(N, H, W, C, device="cuda", generator=g).to(torch.bfloat16)
    s = torch.randn(N, H, W, device="cuda", generator=g)
    tol = 8 * 2.0 ** -24 * np.sqrt(N * H * W) + 2.0 ** -22
    for kind, sign in ((nn.WGRAD_IN1, 1), (nn.WGRAD_OUT1, -1)):
        out = torch.zeros(10, C, device="cuda")
        ws = nn.wgrad_workspace(kind, N, H, W, C, C, "cuda")
        if sign > 0:
            nn._check(lib.sps_nn_conv3x3_in1_wgrad_bias(
                nn._ptr(s), nn._ptr(a), N, H, W, C, nn._ptr(out), nn._ptr(out[9]), nn._ptr(ws),
                ws.numel(), nn._stream()))
            assert torch.allclose(out[9].double(), a.double().sum((0, 1, 2)), rtol=0,
                                  atol=tol * np.sqrt(N * H * W))
        else:
            w = torch.zeros(9, C, device="cuda")
            nn._check(lib.sps_nn_conv3x3_out1_bwd(
                nn._ptr(a), nn._ptr(s), N, H, W, C, nn._ptr(w), None, nn._ptr(out), nn._ptr(ws),
                ws.numel(), nn._stream()))
        for t in range(9):
            v = torch.roll(s, (sign * (1 - t // 3), sign * (1 - t % 3)), dims=(1, 2)).double()
            want = (v[..., None] * a.double()).sum((0, 1, 2))
            # sums of N*H*W unit products
            assert float((out[t].double() - want).abs().max()) <= tol * np.sqrt(N * H * W), (kind, t)


def test_gradients_have_their_own_storage(gpu_lib):
    # a parameter's .grad may be the tensor itself: no two share memory or a
    # version counter
    net = nn.UNet(seed=3).to("cuda")
    x = torch.randn(2, 64, 64, device="cuda")
    net(x).square().sum().backward()
    grads = [p.grad for p in net.parameters()]
    assert len({g.untyped_storage().data_ptr() for g in grads}) == len(grads)
    assert all(g.untyped_storage().nbytes() == 4 * g.numel() for g in grads)
    before = [g._version for g in grads]
    grads[0].add_(1.0)
    assert [g._version for g in grads[1:]] == before[1:]
