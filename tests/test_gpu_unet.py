"""Learned preconditioner kernels against the U-Net oracle (oracle/unet.py).

Single conv: bf16-exact inputs and weights, FP32 accumulation -> within one
bf16 ulp of the oracle (rounded to bf16).  Whole network: against the oracle
run at the same storage precision (``bf16=True``: activations and activation
gradients rounded to bfloat16 where the device stores them; matrix-core
layers with bf16 weights, first/last layers FP32): output within 1e-2
(max-norm relative) and weight gradients within 1e-1 (Frobenius relative)
and 2e-1 (max-norm).  Measured: <= 8e-3 Frobenius for the 2-level network,
up to 6.3e-2 Frobenius / 1.0e-1 max for the deepest decoder layer of the
4-level one -- FP32 accumulation order flips stored values by one bf16 ulp
and ReLU gates near zero, and those flips compound with depth.  An indexing
error gives O(1) differences.  Against the exact FP64 network the same bf16
storage alone moves deep-layer gradients by up to ~20 %, so the exact
comparison is not a useful gate.
"""

import numpy as np
import pytest
import torch

from finitevolx_amd import _lib
from finitevolx_amd import learned as Lm
from oracle import unet as U
from tests.gpu_util import need_gpu

pytestmark = pytest.mark.gpu


def _bf16(t):
    return torch.from_numpy(Lm.to_bf16(t)).to("cuda", torch.bfloat16)


@pytest.mark.parametrize("cin,cout,ups", [(16, 16, False), (32, 48, False), (64, 16, True),
                                          (48, 64, False), (16, 32, True)])
def test_single_conv_mfma(cin, cout, ups):
    need_gpu()
    rng = np.random.default_rng(0)
    Hx, Wx = (12, 40) if ups else (20, 70)
    x = Lm.to_bf16(rng.standard_normal((Hx, Wx, cin))).astype(np.float64)
    w = Lm.to_bf16(rng.standard_normal((3, 3, cout, cin)) * 0.2).astype(np.float64)
    xin = U.up2(x) if ups else x
    ref = U.conv3x3(xin, w)
    got = Lm.conv3x3_bf16(_bf16(x), w, ups=ups).float().cpu().numpy()
    refb = Lm.to_bf16(ref)
    ulp = np.abs(refb).astype(np.float64) * 2.0**-7 + 1e-30
    assert np.all(np.abs(got - refb) <= ulp + 1e-6 * np.abs(ref).max()), np.max(np.abs(got - refb) / ulp)
    got_r = Lm.conv3x3_bf16(_bf16(x), w, ups=ups, relu=True).float().cpu().numpy()
    assert np.all(got_r >= 0) and np.allclose(got_r, np.maximum(got, 0))


@pytest.mark.parametrize("channels", [(16, 32), (16, 32, 48, 64)])
def test_forward_and_gradients_match_oracle(channels):
    need_gpu()
    H = W = 64
    net = Lm.UNet(channels, H, W, seed=1)
    # matrix-core layers run on bf16 weights; the 1-channel edge layers on FP32
    Wt = {k: (v if k in ("e0a", "out") else Lm.to_bf16(v).astype(np.float64))
          for k, v in net.get_weights().items()}
    rng = np.random.default_rng(2)
    x = Lm.to_bf16(rng.standard_normal((H, W))).astype(np.float64)
    ref, cache = U.forward(Wt, x, channels, bf16=True)
    got = net.forward(torch.tensor(x, dtype=torch.float32)).cpu().numpy()
    err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    assert err < 1e-2, err
    gy = rng.standard_normal((H, W))
    gref = U.backward(Wt, cache, gy, channels, bf16=True)
    g = net.grads(torch.tensor(x, dtype=torch.float32), torch.tensor(gy, dtype=torch.float32))
    for k in gref:
        e = np.max(np.abs(g[k] - gref[k])) / max(np.max(np.abs(gref[k])), 1e-30)
        f = np.linalg.norm(g[k] - gref[k]) / max(np.linalg.norm(gref[k]), 1e-30)
        print(f"[unet] {channels} {k}: max {e:.3e} fro {f:.3e}", flush=True)
        assert e < 2e-1 and f < 1e-1, (k, e, f)


def test_training_reduces_loss():
    need_gpu()
    H = W = 32
    net = Lm.UNet((16, 32), H, W, seed=3)
    rng = np.random.default_rng(4)
    xb = torch.tensor(rng.standard_normal((4, H, W)), dtype=torch.float32, device="cuda")
    eb = xb * 0.5  # a learnable linear target
    l0 = net.train_step(xb, eb, 1e-3)
    for _ in range(60):
        l1 = net.train_step(xb, eb, 1e-3)
    assert l1 < 0.5 * l0, (l0, l1)


@pytest.mark.parametrize("channels", [(16,), (32,), (48,), (64,), (16, 32), (32, 64), (64, 48)])
@pytest.mark.parametrize("H,W", [(6, 62), (10, 130)])
def test_weight_gradients_at_tile_edges(channels, H, W):
    """Every (co, ci) block split of the weight-gradient kernel and both
    one-channel layers on fields that end inside a 64 x 4 tile.  Each stored
    tensor on the way to a gradient may differ from the oracle's by one bf16
    ulp (2^-8 relative); there are 4 per level, so the Frobenius distance is
    within 4 * levels * 2^-8.  A tile edge read wrongly moves it by > 0.1."""
    need_gpu()
    net = Lm.UNet(channels, H, W, seed=3)
    Wt = {k: (v if k in ("e0a", "out") else Lm.to_bf16(v).astype(np.float64))
          for k, v in net.get_weights().items()}
    rng = np.random.default_rng(4)
    x = Lm.to_bf16(rng.standard_normal((H, W))).astype(np.float64)
    gy = Lm.to_bf16(rng.standard_normal((H, W))).astype(np.float64)
    _, cache = U.forward(Wt, x, channels, bf16=True)
    ref = U.backward(Wt, cache, gy, channels, bf16=True)
    got = net.grads(torch.tensor(x, device="cuda"), torch.tensor(gy, device="cuda"))
    tol = 4 * len(channels) * 2.0**-8
    for k in ref:
        err = np.linalg.norm(got[k] - ref[k]) / np.linalg.norm(ref[k])
        assert err <= tol, (k, err)


@pytest.mark.parametrize("channels", [(32,), (16, 48), (64,)])
def test_weight_gradients_over_many_tiles(channels):
    """More than 256 tiles on the first level (its blocks hold every output
    channel), fewer on the second (split over the channels), on a plan for a
    larger field; the bound of test_weight_gradients_at_tile_edges."""
    need_gpu()
    H, W = 70, 1030
    net = Lm.UNet(channels, H + 6, W + 70, seed=3)
    Wt = {k: (v if k in ("e0a", "out") else Lm.to_bf16(v).astype(np.float64))
          for k, v in net.get_weights().items()}
    rng = np.random.default_rng(5)
    x = Lm.to_bf16(rng.standard_normal((H, W))).astype(np.float64)
    gy = Lm.to_bf16(rng.standard_normal((H, W))).astype(np.float64)
    _, cache = U.forward(Wt, x, channels, bf16=True)
    ref = U.backward(Wt, cache, gy, channels, bf16=True)
    got = net.grads(torch.tensor(x, device="cuda"), torch.tensor(gy, device="cuda"))
    tol = 4 * len(channels) * 2.0**-8
    for k in ref:
        err = np.linalg.norm(got[k] - ref[k]) / np.linalg.norm(ref[k])
        assert err <= tol, (k, err)


@pytest.mark.parametrize("cin,cout,ups", [(16, 16, False), (48, 32, True), (64, 48, False),
                                          (32, 64, False)])
def test_conv_wide_tiles(cin, cout, ups):
    """Enough rows for the wide tiles (up to 32 output channels; the others take
    16 pixels), whose last column holds 2 pixels and whose last row of tiles 2
    rows; the bound of test_single_conv_mfma."""
    need_gpu()
    rng = np.random.default_rng(1)
    Hx, Wx = (685, 65) if ups else (1370, 130)
    x = Lm.to_bf16(rng.standard_normal((Hx, Wx, cin))).astype(np.float64)
    w = Lm.to_bf16(rng.standard_normal((3, 3, cout, cin)) * 0.2).astype(np.float64)
    ref = U.conv3x3(U.up2(x) if ups else x, w)
    got = Lm.conv3x3_bf16(_bf16(x), w, ups=ups).float().cpu().numpy()
    refb = Lm.to_bf16(ref)
    ulp = np.abs(refb).astype(np.float64) * 2.0**-7 + 1e-30
    assert np.all(np.abs(got - refb) <= ulp + 1e-6 * np.abs(ref).max())


def test_output_layer_gradient_of_a_border_overflow():
    """An activation that overflowed on the field's border counts for the taps
    that reach it from inside and for no others: FP32 sums of the plain formula,
    infinities included.  Activations here are 0 but for one pixel and channel."""
    need_gpu()
    C, H, W = 16, 6, 62
    w = {"e0a": np.zeros((3, 3, C, 1)), "e0b": np.zeros((3, 3, C, C)), "out": np.zeros((3, 3, 1, C))}
    w["e0a"][1, 1, 0, 0] = 1e20
    w["e0b"][1, 1, 0, 0] = 1e20
    for j, i in ((0, 0), (H - 1, W - 1), (0, 30), (2, 31)):
        x = torch.zeros(H, W, device="cuda")
        x[j, i] = 1.0
        net = Lm.UNet((C,), H, W, weights=w)
        got = net.grads(x, torch.ones(H, W, device="cuda"))["out"][:, :, 0, :]
        want = np.zeros((3, 3, C))
        for a in range(3):
            for b in range(3):  # dW[a, b] = sum_p gy[p] d[p + (a - 1, b - 1)]
                if 0 <= j - (a - 1) < H and 0 <= i - (b - 1) < W:
                    want[a, b, 0] = np.inf
        assert np.array_equal(got, want), (j, i, got[:, :, 0])


def test_gradient_slots_come_with_the_first_gradient():
    """A plan that only runs forward holds no slots beyond one layer's; the first
    gradient allocates them, further ones nothing."""
    need_gpu()

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    Lm.UNet((16, 32, 48, 64), 64, 64, seed=0).grads(torch.zeros(64, 64), torch.zeros(64, 64))
    net = Lm.UNet((16, 32, 48, 64), 512, 512, seed=0)
    x = torch.randn(512, 512, device="cuda")
    net.forward(x)
    f0 = free()
    first = net.grads(x, x)
    f1 = free()
    again = net.grads(x, x)
    assert f0 - f1 >= 40 << 20, (f0, f1)
    assert abs(f1 - free()) <= 4 << 20
    for k in first:
        assert np.array_equal(first[k], again[k]), k


@pytest.mark.parametrize("channels", [(16,), (32, 64, 48)])
def test_first_gradient_in_a_graph(channels):
    """A plan's first backward pass may be a captured one (layer by layer in one
    layer's slots); its replays, and eager passes between them, give what a plan
    that never saw a capture gives, bit for bit."""
    need_gpu()
    H, W = 20, 132
    x, gy = (torch.randn(H, W, device="cuda") for _ in range(2))
    ref = Lm.UNet(channels, H, W, seed=1).grads(x, gy)
    net = Lm.UNet(channels, H, W, seed=1)
    flat = torch.zeros(sum(r.size for r in ref.values()), device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _lib.call("fvx_unet_backward_raw", net._h, x.data_ptr(), gy.data_ptr(), H, W,
                  _lib.stream())
    for k in range(4):
        graph.replay()
        _lib.call("fvx_unet_grads", net._h, flat.data_ptr(), 1, _lib.stream())
        got = net._unflatten(flat.cpu().numpy())
        for n in ref:
            assert np.array_equal(got[n], ref[n]), (k, n)
        if k:
            got = net.grads(x, gy)
            for n in ref:
                assert np.array_equal(got[n], ref[n]), (k, n)
