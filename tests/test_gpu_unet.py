"""Learned WFF2 surrogate on the GPU: forward pass and every parameter
gradient of the BF16-MFMA kernels against the FP64 CPU reference
(oracle/unet_ref.py, itself pinned by finite differences), training on GPU
pairs, and the learned DPRA frame with its WFF2 spot check and fallback.

Tolerances: BF16 weights and activations (8-bit mantissa, relative rounding
3.9e-3 per value) through ~15 layers give a few 1e-3 to 1e-2 relative error;
the bars are 3e-2 (forward, relative to the network's correction x - out) and
6e-2 (per-layer relative gradient norm).  The 2-channel input layer's weight
gradient is a sum over pixels of random-phase inputs that cancels to ~1/10 of
its terms, which amplifies the BF16 error it inherits from the whole backward
pass; it is held to direction (cosine > 0.98) and a 0.2 relative norm, which
a wrong tap, channel or sign would fail by far."""
import math

import numpy as np
import pytest

from _util import say

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import glsu  # noqa: E402
from oracle import unet_ref as U  # noqa: E402


def _bf16(a):
    """Round to bfloat16 (nearest even), returned as float64."""
    f = np.ascontiguousarray(a, np.float32)
    u = f.view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32)
    return u.view(np.float32).astype(np.float64)


def _net_and_ref(seed=3, levels=4, base=32):
    net = glsu.UNet(levels, base, seed=seed)
    p = net.params()
    rng = np.random.default_rng(seed)
    p["out.w"] = rng.normal(0, 0.2, p["out.w"].shape).astype(np.float32)
    for k in p:
        if k.endswith(".b"):
            p[k] = rng.normal(0, 0.05, p[k].shape).astype(np.float32)
    net.set_params(p)
    # the CPU reference sees what the kernels use: BF16 weights of the MFMA
    # layers, FP32 weights of the 2-channel input layer and the 1x1 output
    ref = {}
    for k, v in p.items():
        mfma = k.endswith(".w") and not k.startswith("e0a") and not k.startswith("out")
        ref[k] = _bf16(v) if mfma else v.astype(np.float64)
    return net, ref


def _inputs(n, H, W, seed=5):
    rng = np.random.default_rng(seed)
    t = rng.uniform(-np.pi, np.pi, (n, H, W))
    tf = t + rng.normal(0, 0.3, t.shape)
    x = np.exp(1j * t).astype(np.complex64)
    u = np.exp(1j * tf).astype(np.complex64)
    return x, u


def _c2(a):
    return np.stack([a.real, a.imag], -1).astype(np.float64)


def test_forward_matches_cpu_reference():
    net, ref = _net_and_ref()
    x, _ = _inputs(2, 64, 96)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    r = U.forward(ref, _c2(x))
    corr_ref = r - _c2(x)
    err = np.abs(_c2(out) - r).max() / np.abs(corr_ref).max()
    rel = np.linalg.norm(_c2(out) - r) / np.linalg.norm(corr_ref)
    say(f"[unet fwd] max err / max correction = {err:.2e}, relative norm {rel:.2e}")
    assert rel < 3e-2


def test_gradients_match_cpu_reference():
    net, ref = _net_and_ref(seed=4)
    x, u = _inputs(2, 64, 64, seed=6)
    loss = net.loss_grad(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda())
    g = net.grads()
    Lr, gr = U.loss_and_grads(ref, _c2(x), _c2(u))
    say(f"[unet grad] loss gpu {loss:.6f} cpu {Lr:.6f}")
    assert abs(loss - Lr) / Lr < 1e-2
    for k in gr:
        a, b = g[k].astype(np.float64).ravel(), gr[k].ravel()
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
        say(f"   {k:8s} |g|={np.linalg.norm(b):.3e} rel err {rel:.2e} cos {cos:.5f}")
        if k.startswith("e0a"):
            assert rel < 0.2 and cos > 0.98, k
        else:
            assert rel < 6e-2, k


def test_interior_tiles_match_cpu_reference():
    """160 x 224: the full-resolution convs run the persistent 8-row kernel on
    tiles away from the border (unclamped loads from per-thread offsets), on
    border tiles and on a part-width last tile column; forward and every
    gradient against the FP64 reference at the bars above."""
    net, ref = _net_and_ref(seed=8)
    x, u = _inputs(1, 160, 224, seed=9)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    r = U.forward(ref, _c2(x))
    corr_ref = r - _c2(x)
    rel = np.linalg.norm(_c2(out) - r) / np.linalg.norm(corr_ref)
    say(f"[unet fwd 160x224] relative norm {rel:.2e}")
    assert rel < 3e-2
    loss = net.loss_grad(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda())
    g = net.grads()
    Lr, gr = U.loss_and_grads(ref, _c2(x), _c2(u))
    say(f"[unet grad 160x224] loss gpu {loss:.6f} cpu {Lr:.6f}")
    assert abs(loss - Lr) / Lr < 1e-2
    for k in gr:
        a, b = g[k].astype(np.float64).ravel(), gr[k].ravel()
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
        say(f"   {k:8s} rel err {rel:.2e} cos {cos:.5f}")
        if k.startswith("e0a"):
            assert rel < 0.2 and cos > 0.98, k
        else:
            assert rel < 6e-2, k


def test_streamed_weight_tiles_match_cpu_reference():
    """2 x 512 x 1016: the forward convs of more than 64 input channels whose
    16 x 32-pixel tiles give every CU a workgroup stage their weights per
    32-channel chunk in the persistent kernel: the level-1 decoder conv (64 +
    128 upsampled -> 64 channels at 256 x 508, 512 tiles) and the level-2
    128 -> 128 and (128 + 256 upsampled) -> 128 convs (128 x 254, 128 tiles x
    two 64-channel blocks); interior and border tiles, part-width last tile
    columns (28 and 30 pixels).  Forward against the FP64 reference at the bar
    above, per image too."""
    net, ref = _net_and_ref(seed=10)
    x, _ = _inputs(2, 512, 1016, seed=11)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    r = U.forward(ref, _c2(x))
    corr_ref = r - _c2(x)
    rel = np.linalg.norm(_c2(out) - r) / np.linalg.norm(corr_ref)
    rel1 = [np.linalg.norm(_c2(out[i]) - r[i]) / np.linalg.norm(corr_ref[i]) for i in range(2)]
    say(f"[unet fwd 2x512x1016] relative norm {rel:.2e} (per image {rel1[0]:.2e}, {rel1[1]:.2e})")
    assert rel < 3e-2 and max(rel1) < 3e-2


@pytest.mark.parametrize("levels,base,shape", [(3, 64, (1, 64, 96)), (2, 32, (2, 48, 80))])
def test_other_depths_and_widths_match_cpu_reference(levels, base, shape):
    """Networks other than 4 levels x 32 channels: with 64 base channels the
    full-resolution convs run on the 64-channel kernels (the first encoder's
    max-pool from a conv epilogue) and the output layer sums 64 channels;
    with 2 levels a single pooling step.  Forward and every gradient against
    the FP64 reference at the bars above."""
    net, ref = _net_and_ref(seed=12, levels=levels, base=base)
    n, H, W = shape
    x, u = _inputs(n, H, W, seed=13)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    r = U.forward(ref, _c2(x), levels=levels)
    corr_ref = r - _c2(x)
    rel = np.linalg.norm(_c2(out) - r) / np.linalg.norm(corr_ref)
    say(f"[unet fwd L{levels} b{base} {shape}] relative norm {rel:.2e}")
    assert rel < 3e-2
    loss = net.loss_grad(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda())
    g = net.grads()
    Lr, gr = U.loss_and_grads(ref, _c2(x), _c2(u), levels=levels)
    say(f"[unet grad L{levels} b{base}] loss gpu {loss:.6f} cpu {Lr:.6f}")
    assert abs(loss - Lr) / Lr < 1e-2
    for k in gr:
        a, b = g[k].astype(np.float64).ravel(), gr[k].ravel()
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
        say(f"   {k:8s} rel err {rel:.2e} cos {cos:.5f}")
        if k.startswith("e0a"):
            assert rel < 0.2 and cos > 0.98, k
        else:
            assert rel < 6e-2, k


def test_training_reduces_loss():
    x, u = glsu.learned.make_pairs(nseq=1, nframes=3, size=256, seed0=777)
    net = glsu.UNet(4, 32, seed=1)
    losses = glsu.learned.train(net, x, u, crops=4 * 80, batch=4, crop=128, lr=2e-3, seed=0,
                                log=say, log_every=20)
    first, last = np.mean(losses[:5]), np.mean(losses[-5:])
    say(f"[unet train] loss {first:.4f} -> {last:.4f}")
    assert np.isfinite(losses).all()
    assert last < 0.7 * first


def test_learned_frame_fallback_and_net_paths():
    W = H = 256
    frames = glsu.gen_frames(W, H, 2, 42)
    phi0 = glsu.synth.phase(W, H, 3.0, 0.05)
    net = glsu.UNet(4, 32, seed=2)
    # plain reference
    d0 = glsu.DPRA(phi0)
    ref = d0(frames).cpu().numpy()
    # tol = 0: every frame falls back to WFF2 -> identical to the plain chain
    d1 = glsu.DPRA(phi0)
    outs = []
    for t in range(2):
        res, fb = d1.frame_learned(frames[t], net, tol=0.0, tile=(96, 96))
        d1.update_ref_phi()
        outs.append(d1.last_dphi.cpu().numpy())
        say(f"[learned] tol 0 frame {t}: residual {res:.3e} fallback {fb}")
        assert fb and res > 0
    assert np.array_equal(np.stack(outs), ref)
    # asynchronous calls: the decision stays on the device; tol 0 -> every
    # frame falls back, identical to the plain chain, and the statistics count it
    d3 = glsu.DPRA(phi0)
    outs3 = []
    for t in range(2):
        assert d3.frame_learned(frames[t], net, tol=0.0, tile=(32, 160), sync=False) is None
        d3.update_ref_phi()
        outs3.append(d3.last_dphi.cpu().numpy())
    assert np.array_equal(np.stack(outs3), ref)
    st = d3.learned_stats()
    say(f"[learned] async stats {st}")
    assert st["frames"] == 2 and st["fallbacks"] == 2 and st["max_rms"] > 0
    # spot checks at the corners: the window is clipped by the image border
    for tile in [(0, 0), (W - 64, H - 64), (0, H - 64)]:
        res, fb = glsu.DPRA(phi0).frame_learned(frames[0], net, tol=1e9, tile=tile)
        say(f"[learned] corner tile {tile}: residual {res:.3e}")
        assert 0 < res < 10 and not fb
    # untrained net = identity (out = z): no check -> the update uses angle(z)
    d2 = glsu.DPRA(phi0)
    res, fb = d2.frame_learned(frames[0], net, tol=-1.0)
    assert res == -1.0 and not fb
    z = d2.last_z()
    zn = d2.last_net()
    assert torch.equal(z, zn)
    dphi = d2.last_dphi.cpu().numpy()
    expect = np.angle(z.cpu().numpy())
    assert np.abs(np.angle(np.exp(1j * (dphi - expect)))).max() < 1e-6


@pytest.mark.parametrize("levels,base,n,H,W", [
    (2, 32, 1, 8, 34),    # two rows of strips less than one workgroup; a 2-pixel remainder
    (2, 32, 3, 24, 130),  # chunks that cross image borders; a strip of 2 pixels in a second block
    (2, 96, 1, 16, 66),   # channel counts that only 32 divides
    (3, 64, 2, 16, 260),  # 64-channel tiles on both sources of the decoder convs; 4-row bottom
])
def test_gradients_at_strip_and_chunk_edges(levels, base, n, H, W):
    """The weight-gradient kernels walk 32-pixel strips and chunks of rows
    across the images of a batch: widths that leave part strips, heights that
    split unevenly, every channel tile.  Bars as above (the same BF16
    rounding enters)."""
    net, ref = _net_and_ref(seed=21, levels=levels, base=base)
    x, u = _inputs(n, H, W, seed=22)
    loss = net.loss_grad(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda())
    g = net.grads()
    Lr, gr = U.loss_and_grads(ref, _c2(x), _c2(u), levels)
    assert abs(loss - Lr) / Lr < 1e-2
    for k in gr:
        a, b = g[k].astype(np.float64).ravel(), gr[k].ravel()
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
        say(f"   {k:8s} rel err {rel:.2e} cos {cos:.5f}")
        if k.startswith("e0a"):
            assert rel < 0.2 and cos > 0.98, k
        else:
            assert rel < 6e-2, k


@pytest.mark.parametrize("levels,base,H,W", [
    (2, 32, 16, 130),   # 130 = 128 + 2 pixels of a strip group, 2 * 64 + 2 of the input layer's lanes
    (2, 32, 16, 260),   # the half-resolution layers have the 2-pixel remainder too
    (2, 64, 16, 66),    # 64-channel tiles: strips of 64 pixels
    (2, 96, 16, 130),   # channel counts that only 32 divides
])
def test_gradients_of_a_signal_in_the_last_columns(levels, base, H, W):
    """The target differs from the output in the last two columns only, so
    every layer's gradient comes from the part strips there.  Bar: a lost
    remainder changes the layer it belongs to by at least 0.48 in norm (the
    FP64 reference with those columns of the layer's gradient left out); BF16
    rounding of activations and gradients, emulated in the reference, by at
    most 0.16 over four seeds (few pixels: ReLU and pooling decisions weigh
    more than in the tests above)."""
    net, ref = _net_and_ref(seed=31, levels=levels, base=base)
    x, _ = _inputs(1, H, W, seed=32)
    rng = np.random.default_rng(33)
    delta = np.zeros((1, H, W), np.complex64)
    delta[:, :, -2:] = rng.normal(0, 0.5, (1, H, 2)) + 1j * rng.normal(0, 0.5, (1, H, 2))
    xg = torch.from_numpy(x).cuda()
    net.loss_grad(xg, net.forward(xg) + torch.from_numpy(delta).cuda())
    g = net.grads()
    _, gr = U.loss_and_grads(ref, _c2(x), U.forward(ref, _c2(x), levels) + _c2(delta), levels)
    for k in gr:
        a, b = g[k].astype(np.float64).ravel(), gr[k].ravel()
        rel = np.linalg.norm(a - b) / np.linalg.norm(b)
        say(f"   {k:8s} rel err {rel:.2e}")
        assert rel < 0.3, k


def test_gradients_with_several_strips_per_workgroup():
    """288 and 576 channels on 8 x 832 pixels: more strips than workgroups a
    channel tile, so each workgroup walks several, for all three tile shapes
    (32 x 32: 288 -> 288 and 864 -> 288, 64 x 32: 288 -> 576, 64 x 64: 576 ->
    576).  Bars as above."""
    levels, base, H, W = 2, 288, 8, 832
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for cout, cin, mb, nb, strip, wgs, w in [(288, 288, 1, 1, 128, 2 * cus, W),
                                             (288, 864, 1, 1, 128, 2 * cus, W),
                                             (576, 288, 2, 1, 128, cus, W // 2),
                                             (576, 576, 2, 2, 64, cus, W // 2)]:
        assert -(-w // strip) > wgs // (cout // (32 * mb) * (cin // (32 * nb)))
    net, ref = _net_and_ref(seed=41, levels=levels, base=base)
    x, u = _inputs(1, H, W, seed=42)
    loss = net.loss_grad(torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda())
    g = net.grads()
    Lr, gr = U.loss_and_grads(ref, _c2(x), _c2(u), levels)
    assert abs(loss - Lr) / Lr < 1e-2
    for k in gr:
        a, b = g[k].astype(np.float64).ravel(), gr[k].ravel()
        rel = np.linalg.norm(a - b) / np.linalg.norm(b)
        say(f"   {k:8s} rel err {rel:.2e}")
        assert rel < (0.2 if k.startswith("e0a") else 6e-2), k


def test_gradients_repeat_bit_for_bit():
    """Every gradient sum runs in a fixed order: the same inputs give the same
    bits, also after a step on another shape (other buffers)."""
    net, _ = _net_and_ref(seed=51, levels=3)
    x, u = (torch.from_numpy(a).cuda() for a in _inputs(3, 48, 132, seed=52))
    x2, u2 = (torch.from_numpy(a).cuda() for a in _inputs(1, 16, 260, seed=53))
    first = (net.loss_grad(x, u), net.get_flat(grads=True))
    net.loss_grad(x2, u2)
    for _ in range(3):
        loss = net.loss_grad(x, u)
        assert loss == first[0] and np.array_equal(net.get_flat(grads=True), first[1])


def test_seeded_weights_are_the_standard_normal_draws():
    """A network made from a seed has He-normal weights drawn layer by layer
    from the 64-bit Mersenne twister by the polar method, second coordinate
    first (what std::normal_distribution<double> of libstdc++ draws), zero
    biases and a zero output layer."""
    M = (1 << 64) - 1

    class Twister:
        def __init__(self, seed):
            self.s, self.i = [seed & M], 312
            for k in range(1, 312):
                p = self.s[-1]
                self.s.append((6364136223846793005 * (p ^ (p >> 62)) + k) & M)

        def __call__(self):
            if self.i == 312:
                s = self.s
                for k in range(312):
                    y = (s[k] & ~0x7FFFFFFF & M) | (s[(k + 1) % 312] & 0x7FFFFFFF)
                    s[k] = s[(k + 156) % 312] ^ (y >> 1) ^ (0xB5026F5AA96619E9 if y & 1 else 0)
                self.i = 0
            y = self.s[self.i]
            self.i += 1
            y ^= (y >> 29) & 0x5555555555555555
            y ^= (y << 17) & 0x71D67FFFEDA60000
            y ^= (y << 37) & 0xFFF7EEE000000000
            return y ^ (y >> 43)

    for seed in (0, 12345678901234567890):
        p = glsu.UNet(2, 32, seed=seed).params()
        rng = Twister(seed)

        def unit():
            return 2.0 * min(float(rng()) / 2.0 ** 64, math.nextafter(1.0, 0.0)) - 1.0

        for name, kind, ci, co in glsu.learned.layer_specs(2, 32):
            assert not p[name + ".b"].any()
            if name == "out":
                assert not p[name + ".w"].any()
                continue
            sd, want = math.sqrt(2.0 / (9 * ci)), []
            for _ in range(0, 9 * ci * co, 2):
                while True:
                    a, b = unit(), unit()
                    r2 = a * a + b * b
                    if 0.0 < r2 <= 1.0:
                        break
                m = math.sqrt(-2.0 * math.log(r2) / r2)
                want += [b * m * sd, a * m * sd]
            assert np.array_equal(p[name + ".w"].ravel(), np.float32(want)), (seed, name)
