"""GPU parity of the learned restoration stage against the FP64 oracle
(oracle/unet_ref.py, with bf16 rounding at the GPU's storage points).

Tolerances: a bf16 output may differ from the oracle's rounding by one bf16
step (relative 2^-7 at most) where FP32 and FP64 accumulation round differently;
FP32 outputs (weight gradients, the network output) are compared in relative
L2 norm.
"""
import os

import numpy as np
import pytest
import torch

from oracle import unet_ref as U
from recview_amd import unet as RU

pytestmark = pytest.mark.gpu
DEV = "cuda"
WEIGHTS = os.path.join(os.path.dirname(RU.__file__), "weights", "unet_sparse8.npz")


def bf(a):
    """numpy -> int16 device tensor of bf16 bits (round to nearest even)."""
    return RU.to_bf16_bits(torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV)).contiguous()


def unbf(t):
    return RU.from_bf16_bits(t).double().cpu().numpy()


def assert_bf16_close(got, ref):
    bound = 2.0 ** -7 * np.abs(ref) + 1e-6 * np.abs(ref).max()   # one bf16 step
    bad = np.abs(got - ref) > bound
    assert not bad.any(), (int(bad.sum()), float(np.abs(got - ref).max()))
    # one-step differences are rare rounding ties, not systematic
    assert np.mean(got != ref) < 0.02


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("cin,cout,H,W,relu", [(32, 32, 16, 16, True), (64, 32, 12, 20, False),
                                               (96, 64, 8, 32, True), (32, 128, 24, 16, True),
                                               (384, 128, 8, 16, True), (128, 256, 5, 7, True)])
def test_conv_forward(cin, cout, H, W, relu):
    rng = np.random.default_rng(cin + cout + H)
    B = 2
    x = U.bf16_round(rng.standard_normal((B, H, W, cin)))
    w = rng.standard_normal((cout, 3, 3, cin)) * np.sqrt(2.0 / (9 * cin))
    b = rng.standard_normal(cout) * 0.1
    out = RU.conv3x3(bf(x), torch.from_numpy(w).float().to(DEV), torch.from_numpy(b).float().to(DEV),
                     cin, cout, relu=relu, shape=(B, H, W))
    torch.cuda.synchronize()
    ref = U.conv3x3(x, U.bf16_round(w.astype(np.float32)), b.astype(np.float32))
    ref = U.bf16_round(np.maximum(ref, 0) if relu else ref)
    assert_bf16_close(unbf(out), ref)


def test_conv_channel_slices():
    """Input and output as channel slices of wider tensors (the concat layout)."""
    rng = np.random.default_rng(5)
    B, H, W = 1, 16, 32
    big = U.bf16_round(rng.standard_normal((B, H, W, 96)))
    w = rng.standard_normal((32, 3, 3, 32)) * 0.1
    out = bf(np.full((B, H, W, 96), 7.0))
    RU.conv3x3(bf(big), torch.from_numpy(w).float().to(DEV), None, 32, 32, relu=False, in_stride=96, in_off=64,
               out=out, out_stride=96, out_off=32, shape=(B, H, W))
    torch.cuda.synchronize()
    got = unbf(out)
    ref = U.bf16_round(U.conv3x3(big[..., 64:], U.bf16_round(w.astype(np.float32))))
    assert_bf16_close(got[..., 32:64], ref)
    assert (got[..., :32] == 7.0).all() and (got[..., 64:] == 7.0).all()


@pytest.mark.parametrize("cin,cout", [(96, 32), (64, 64), (256, 128)])
def test_conv_data_gradient_with_mask(cin, cout):
    rng = np.random.default_rng(cin)
    B, H, W = 2, 8, 16
    g = U.bf16_round(rng.standard_normal((B, H, W, cout)))
    m = U.bf16_round(rng.standard_normal((B, H, W, cin)))
    w = rng.standard_normal((cout, 3, 3, cin)) * 0.1
    out = RU.conv3x3(bf(g), torch.from_numpy(w).float().to(DEV), None, cin, cout, relu=False, mask=bf(m),
                     mask_stride=cin, data_gradient=True, shape=(B, H, W))
    torch.cuda.synchronize()
    ref = U.bf16_round((m > 0) * U.conv3x3_dgrad(g, U.bf16_round(w.astype(np.float32))))
    assert_bf16_close(unbf(out), ref)


@pytest.mark.parametrize("cin,cout,H,W", [(32, 32, 16, 16), (96, 32, 24, 32), (64, 128, 8, 16),
                                          (256, 256, 8, 8), (32, 64, 12, 20)])
def test_conv_weight_gradient(cin, cout, H, W):
    rng = np.random.default_rng(cin * 7 + cout)
    B = 3
    g = U.bf16_round(rng.standard_normal((B, H, W, cout)))
    x = U.bf16_round(rng.standard_normal((B, H, W, cin)))
    dw, db = RU.conv3x3_wgrad(bf(g), bf(x), cin, cout, (B, H, W))
    torch.cuda.synchronize()
    rw, rb = U.conv3x3_wgrad(g, x)
    assert rel(dw.double().cpu().numpy(), rw) < 1e-5
    assert rel(db.double().cpu().numpy(), rb) < 1e-5


@pytest.mark.parametrize("cin,cout,B,H,W", [
    (32, 32, 1, 2, 2),           # one patch, mostly empty
    (64, 32, 1, 9, 17),          # one row and one column past a patch
    (32, 32, 3, 130, 325),       # 1071 patches for 1024 splits: some splits walk two
    (256, 256, 2, 41, 63),       # 32 splits of 48 patches
    (32, 64, 1, 200, 24)])       # 16 to 127 splits
def test_conv_weight_gradient_splits(cin, cout, B, H, W):
    """Patch remainders and split counts of the weight gradient against the FP64 oracle:
    FP32 sums of at most 65000 products, rounding errors of random sign, so well below
    sqrt(65000) / 2 * 2^-24 = 7.6e-6 of the result's RMS."""
    rng = np.random.default_rng(cin + cout + H)
    g = U.bf16_round(rng.standard_normal((B, H, W, cout)))
    x = U.bf16_round(rng.standard_normal((B, H, W, cin)))
    dw, db = RU.conv3x3_wgrad(bf(g), bf(x), cin, cout, (B, H, W))
    torch.cuda.synchronize()
    rw, rb = U.conv3x3_wgrad(g, x)
    assert rel(dw.double().cpu().numpy(), rw) < 1e-5
    assert rel(db.double().cpu().numpy(), rb) < 1e-5


def _images(rng, B, H, W):
    """Smooth random images with edges, like reconstructed slices."""
    x = rng.standard_normal((B, H, W))
    k = np.ones(5) / 5
    for ax in (1, 2):
        x = np.apply_along_axis(lambda v: np.convolve(v, k, mode="same"), ax, x)
    return x + (x > 0.2)


def test_network_forward_matches_oracle():
    net = RU.Unet(32, 4, seed=3)
    p = net.get_params().astype(np.float64)
    rng = np.random.default_rng(0)
    x = _images(rng, 2, 32, 48)
    scale = 1.7
    got = net.forward(torch.from_numpy(x).float().to(DEV).contiguous(), scale)
    torch.cuda.synchronize()
    x32 = x.astype(np.float32).astype(np.float64)
    y, _ = U.UnetRef(32, 4).forward(p, x32, scale)
    y64, _ = U.UnetRef(32, 4).forward(p, x32, scale, rnd=None)
    res = got.double().cpu().numpy() - x32
    # Per layer the GPU matches the bf16-emulating oracle to rare one-step
    # flips (test_conv_*).  Through 15 layers a flip shifts later values by a
    # fraction of a bf16 step, which re-decides later roundings, so the two
    # agree to the size of the bf16 rounding noise itself (emulated vs exact
    # network, ~1 %) and no closer; a wrong term or index would be O(1).
    e_emul = rel(res, y / scale - x32)
    noise = rel(y / scale - x32, y64 / scale - x32)
    assert e_emul < 1.5e-2 and e_emul < 1.5 * noise, (e_emul, noise)
    net.close()


def test_inference_forward_equals_training_forward():
    """Inference lets each decoder convolution read its upsampled half in place;
    the training forward materialises the concatenation.  Same arithmetic, so
    with a zero target the training loss mean(y^2) equals that of the
    inference output."""
    net = RU.Unet(32, 4, seed=7)
    rng = np.random.default_rng(3)
    x = torch.from_numpy(_images(rng, 2, 32, 48).astype(np.float32)).to(DEV)
    out = net.forward(x, 1.0)
    torch.cuda.synchronize()
    y = out.double().cpu().numpy()
    loss, _ = net.loss_grad(x, torch.zeros_like(x), 1.0)
    ref = float(np.mean(y * y))
    assert abs(loss - ref) <= 1e-6 * ref, (loss, ref)
    net.close()


def test_fused_edge_convolution_bit_identical(monkeypatch):
    """Inference computes the edge convolution inside the first 32 -> 32
    convolution's launch (same operation order); the network output equals the
    two-launch form bit for bit, on shapes whose 16 x 16 patches do not divide
    the image or fill the last block of four patches, and a batch of three."""
    net = RU.Unet(32, 4, seed=11)
    rng = np.random.default_rng(5)
    for (B, H, W) in ((3, 40, 56), (1, 24, 200), (2, 136, 72)):
        x = torch.from_numpy(_images(rng, B, H, W).astype(np.float32)).to(DEV).contiguous()
        fused = net.forward(x, 1.3).clone()
        torch.cuda.synchronize()
        monkeypatch.setenv("RECVIEW_UNET_FUSED", "0")
        split = net.forward(x, 1.3).clone()
        torch.cuda.synchronize()
        monkeypatch.delenv("RECVIEW_UNET_FUSED")
        assert torch.equal(fused, split), (B, H, W, (fused - split).abs().max().item())
        assert fused.abs().max().item() > 0
    net.close()


def test_network_gradients_match_oracle():
    net = RU.Unet(32, 4, seed=4)
    rng = np.random.default_rng(1)
    p = net.get_params().astype(np.float64)
    p[np.concatenate([np.arange(b, b + co) for _, _, co, _, b in RU.param_layout()])] = \
        rng.standard_normal(sum(co for _, _, co, _, _ in RU.param_layout())) * 0.05
    net.set_params(p.astype(np.float32))
    x = _images(rng, 2, 32, 32).astype(np.float32)
    t = (x + 0.3 * rng.standard_normal(x.shape)).astype(np.float32)
    scale = 0.8
    loss, g = net.loss_grad(torch.from_numpy(x).to(DEV), torch.from_numpy(t).to(DEV), scale)
    rl, rg = U.UnetRef(32, 4).loss_grad(p.astype(np.float32).astype(np.float64), x, t, scale)
    assert abs(loss - rl) <= 1e-4 * rl
    for name, cin, cout, w, b in RU.param_layout():
        gw, rw = g[w:w + 9 * cin * cout].astype(np.float64), rg[w:w + 9 * cin * cout]
        gb, rb = g[b:b + cout].astype(np.float64), rg[b:b + cout]
        assert rel(gw, rw) < 2e-2, (name, rel(gw, rw))
        assert rel(gb, rb) < 2e-2, (name, rel(gb, rb))
    net.close()


@pytest.mark.parametrize("base,B,H,W", [(32, 1, 2, 2), (32, 3, 10, 66), (32, 1, 16, 64), (64, 2, 18, 34), (64, 1, 6, 70)])
def test_edge_layer_gradients_sizes(base, B, H, W):
    """Gradients of the first and last layer around the strips of their kernel (64 or 32
    columns x 8 rows).  The layers between copy their channels (one centre tap) and the
    numbers are small integers, so every activation is exact in bf16 and no ReLU sits on
    a rounding: the last layer's gradients are FP32 sums (1e-5), the first layer's
    terms carry one bf16 rounding of 2^-9 each (2^-7 of the whole)."""
    print(f"case base={base} {B}x{H}x{W}", flush=True)
    rng = np.random.default_rng(H * W)
    layout = {name: (ci, co, w, b) for name, ci, co, w, b in RU.param_layout(base, 2)}
    net = RU.Unet(base, 2, seed=6)
    p = np.zeros_like(net.get_params())
    for name in ("enc0b", "dec0a", "dec0b"):
        ci, co, w, _ = layout[name]
        k = p[w:w + 9 * ci * co].reshape(co, 9, ci)
        first = ci - base                                   # dec0a: the skip's channels come last
        for c in range(co):
            k[c, 4, first + c] = 1
    ci, co, w, b = layout["enc0a_in"]
    p[w:w + 9 * co] = rng.integers(-2, 3, 9 * co)
    p[b:b + co] = rng.integers(0, 3, co)
    ci, co, w, b = layout["out"]
    p[w:w + 9 * ci] = rng.integers(-1, 2, 9 * ci)
    net.set_params(p)
    x = rng.integers(-2, 3, (B, H, W)).astype(np.float32)
    t = rng.integers(-3, 4, (B, H, W)).astype(np.float32)
    loss, g = net.loss_grad(torch.from_numpy(x).to(DEV), torch.from_numpy(t).to(DEV), 1.0)
    rl, rg = U.UnetRef(base, 2).loss_grad(p.astype(np.float64), x, t, 1.0)
    assert abs(loss - rl) <= 1e-5 * rl
    for name, tol in (("out", 1e-5), ("enc0a_in", 2.0 ** -7)):
        ci, co, w, b = layout[name]
        assert rel(g[w:w + 9 * ci * co], rg[w:w + 9 * ci * co]) <= tol, name
        assert rel(g[b:b + co], rg[b:b + co]) <= tol, name
    net.close()


def test_training_reduces_loss():
    """Adam on a fixed batch: the network learns a 3x3 blur of its input."""
    net = RU.Unet(32, 4, seed=5)
    rng = np.random.default_rng(2)
    x = _images(rng, 4, 64, 64).astype(np.float32)
    t = x.copy()
    t[:, 1:-1, 1:-1] = sum(x[:, 1 + dy:x.shape[1] - 1 + dy, 1 + dx:x.shape[2] - 1 + dx]
                           for dy in (-1, 0, 1) for dx in (-1, 0, 1)) / 9
    xg, tg = torch.from_numpy(x).to(DEV), torch.from_numpy(t).to(DEV)
    losses = [net.train_step(xg, tg, 1.0, 1e-3) for _ in range(60)]
    assert losses[-1] < 0.3 * losses[0], (losses[0], losses[-1])
    net.close()


def test_shape_errors_raise():
    net = RU.Unet(32, 4, seed=6)
    x = torch.zeros(1, 20, 32, device=DEV)
    with pytest.raises(RuntimeError, match="divisible"):
        net.forward(x, 1.0)
    net.close()


@pytest.mark.skipif(not os.path.exists(WEIGHTS), reason="trained weights not present")
def test_trained_network_restores_sparse_view():
    """Held-out phantoms: sparse-view (1/8 angles) FBP + the trained network is
    much closer to full-angle FBP, and to the phantom, than sparse FBP alone."""
    from recview_amd import learned
    net = RU.Unet.load(WEIGHTS)
    res = learned.evaluate(net, net.scale, [2_000_001, 2_000_002])
    s = learned.summarize(res)
    print(s)
    assert s["psnr_vs_full"]["restored"] > s["psnr_vs_full"]["sparse"] + 3.0
    assert s["psnr_phantom"]["restored"] > s["psnr_phantom"]["sparse"] + 1.0
    assert s["ssim_vs_full"]["restored"] > s["ssim_vs_full"]["sparse"]
    net.close()


@pytest.mark.parametrize("W", [64, 70])
def test_edge_layer_gradients_of_an_infinite_target(W):
    """A target that is infinite in the last column reaches the last layer's weights of
    the taps that see that pixel from inside the image, and no others, also where the
    kernel's strips of 64 columns end past the image."""
    B, H = 1, 12
    rng = np.random.default_rng(W)
    net = RU.Unet(32, 2, seed=8)
    x = torch.from_numpy(rng.standard_normal((B, H, W)).astype(np.float32)).to(DEV)
    t = torch.zeros_like(x)
    t[0, 5, W - 1] = float("inf")
    _, g = net.loss_grad(x, t, 1.0)
    net.close()
    layout = {name: (ci, co, w, b) for name, ci, co, w, b in RU.param_layout(32, 2)}
    ci, co, w, b = layout["out"]
    taps = np.isfinite(g[w:w + 9 * ci].reshape(3, 3, ci))
    assert taps[:, 2].all()                            # the neighbour to the right is outside
    assert not taps[:, :2].all()


@pytest.mark.parametrize("cin,cout,B,H,W", [
    (128, 128, 1, 8, 16), (128, 64, 1, 17, 33), (128, 128, 2, 40, 70),    # four waves share a column's parts
    (256, 128, 1, 8, 8), (512, 256, 1, 9, 40), (256, 128, 3, 70, 90)])    # one does
def test_conv_weight_gradient_sums_of_wide_layers(cin, cout, B, H, W):
    """The sums of a wide layer's weight-gradient parts, from one part to as many as the
    layer takes, against the FP64 oracle (FP32 sums of at most 18900 products: well below
    sqrt(18900) / 2 * 2^-24 = 4.1e-6 of the result's RMS)."""
    rng = np.random.default_rng(cin + cout + H)
    g = U.bf16_round(rng.standard_normal((B, H, W, cout)))
    x = U.bf16_round(rng.standard_normal((B, H, W, cin)))
    dw, db = RU.conv3x3_wgrad(bf(g), bf(x), cin, cout, (B, H, W))
    torch.cuda.synchronize()
    rw, rb = U.conv3x3_wgrad(g, x)
    assert rel(dw.double().cpu().numpy(), rw) < 1e-5
    assert rel(db.double().cpu().numpy(), rb) < 1e-5
