"""GPU parity: libglsu (HIP, FP32) against the FP64 CPU oracle on the same inputs.

Bars: wrapped phase error of the DPRA chain <= 1e-3 rad RMS per
frame.  Isolated WFF2 on identical inputs: relative field error <= 1e-4 and
phase error <= 1e-4 rad RMS.  DPRA least squares alone: <= 1e-4 rad RMS.
"""
import numpy as np
import pytest

from _util import say, wrapped_err

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import glsu  # noqa: E402


def _seq(O, W, H, T, seed, **kw):
    frames, phi0 = O.gen_sequence(W, H, T, seed, dtype=np.float32, **kw)
    return frames, phi0


@pytest.mark.parametrize("W,H,sig,lo,hi,st", [
    (256, 256, 10.0, -0.2, 0.2, 0.1),
    (200, 180, 10.0, -0.2, 0.2, 0.1),
    (64, 48, 2.0, -0.6, 0.6, 0.3),
    (371, 366, 10.0, -0.2, 0.2, 0.1),
])
def test_wft2_matches_oracle(oracle, W, H, sig, lo, hi, st):
    say(f"[wft2] {W}x{H} sigma={sig} grid=({lo},{hi},{st})")
    frames, phi0 = _seq(oracle, W, H, 2, seed=11)
    od = oracle.DPRA(phi0, sigx=sig, wxl=lo, wxh=hi, wxi=st)
    f = od.ls(frames[1].astype(np.float64)).astype(np.complex64)
    ref = oracle.WFF2(W, H, sig, lo, hi, st)(f.astype(np.complex128))
    w = glsu.WFT2(W, H, params=glsu.wff_params(sig, lo, hi, st))
    out = w(torch.from_numpy(f).cuda()).cpu().numpy()
    torch.cuda.synchronize()
    rel = np.abs(out - ref).max() / np.abs(ref).max()
    rms, mx = wrapped_err(np.angle(out), np.angle(ref))
    say(f"   rel={rel:.3e} phase rms={rms:.3e} max={mx:.3e} thr={w.info()['thr']:.6f}")
    assert rel < 1e-4
    assert rms < 1e-4


@pytest.mark.parametrize("W,H,x,y", [
    (300, 190, (6.0, -0.4, 0.4, 0.2), (12.0, -0.1, 0.2, 0.1)),
    (150, 260, (14.0, -0.15, 0.15, 0.05), (4.0, -0.6, 0.3, 0.3)),
])
def test_wft2_asymmetric_windows_match_oracle(oracle, W, H, x, y):
    """Different window width, frequency range and step along x and y: the
    row and column plans, padded lengths and window spectra differ per axis
    (the oracle is pinned for this case by the brute-force convolution)."""
    say(f"[wft2 asym] {W}x{H} x={x} y={y}")
    frames, phi0 = _seq(oracle, W, H, 2, seed=17)
    od = oracle.DPRA(phi0)
    f = od.ls(frames[1].astype(np.float64)).astype(np.complex64)
    ref = oracle.WFF2(W, H, x[0], x[1], x[2], x[3], sigy=y[0], wyl=y[1], wyh=y[2],
                      wyi=y[3])(f.astype(np.complex128))
    w = glsu.WFT2(W, H, params=glsu.wff_params(x[0], x[1], x[2], x[3], sigma_y=y[0], wyl=y[1],
                                               wyh=y[2], wyi=y[3]))
    out = w(torch.from_numpy(f).cuda()).cpu().numpy()
    torch.cuda.synchronize()
    rel = np.abs(out - ref).max() / np.abs(ref).max()
    rms, mx = wrapped_err(np.angle(out), np.angle(ref))
    say(f"   rel={rel:.3e} phase rms={rms:.3e} max={mx:.3e} thr={w.info()['thr']:.6f}")
    assert rel < 1e-4
    assert rms < 1e-4


@pytest.mark.parametrize("W,H", [(256, 256), (1024, 1024), (77, 53)])
def test_dpra_ls_matches_oracle(oracle, W, H):
    say(f"[dpra-ls] {W}x{H}")
    frames, phi0 = _seq(oracle, W, H, 2, seed=5)
    od = oracle.DPRA(phi0)
    zref = od.ls(frames[1].astype(np.float64))
    d = glsu.DPRA(phi0)
    d.dpra_per_frame(torch.from_numpy(frames[1]).cuda())
    z = d.last_z().cpu().numpy()
    rms, mx = wrapped_err(np.angle(z), np.angle(zref))
    say(f"   z phase rms={rms:.3e} max={mx:.3e}  |z|-1 max={np.abs(np.abs(z) - 1).max():.2e}")
    assert rms < 1e-4
    assert mx < 1e-2


@pytest.mark.parametrize("W,H,T,amp0,amp1,carrier", [
    (1024, 1024, 3, 3.0, 0.1, 0.05),      # the C2 settings, first frames
    (256, 256, 20, 1.0, 0.02, 0.15),      # carrier dominates the peaks gradient
    (512, 384, 8, 3.0, 0.1, 0.05),
])
def test_dpra_chain_matches_oracle(oracle, W, H, T, amp0, amp1, carrier):
    """Well-conditioned sequences (the local fringe frequency stays away from
    zero): strict bar, <= 1e-3 rad RMS on every frame."""
    say(f"[chain] {W}x{H} T={T} amp=({amp0},{amp1}) carrier={carrier}")
    frames, phi0 = _seq(oracle, W, H, T, seed=7, amp0=amp0, amp1=amp1, carrier=carrier)
    ref = oracle.DPRA(phi0).run(frames.astype(np.float64))
    out = glsu.DPRA(phi0)(torch.from_numpy(frames).cuda()).cpu().numpy()
    for t in range(T):
        rms, mx = wrapped_err(out[t], ref[t])
        say(f"   frame {t}: rms={rms:.3e} max={mx:.3e}")
        assert rms < 1e-3


def test_graph_equals_eager(oracle):
    """hipGraph replays of the frame chain equal the eager chain bit for bit;
    the same handle replays its captured graphs (calls 3 and 4), with eager
    work and synchronisation between the replays."""
    W, H, T = 192, 160, 6
    say(f"[graph] {W}x{H} T={T}")
    frames, phi0 = _seq(oracle, W, H, T, seed=3)
    fr = torch.from_numpy(frames).cuda()
    e = glsu.DPRA(phi0)
    g = glsu.DPRA(phi0)
    for rep in range(4):
        say(f"   call {rep}")
        a = e(fr).cpu()
        b = g(fr, graph=True).cpu()
        torch.cuda.synchronize()
        assert torch.equal(a, b), f"call {rep}: max diff {(a - b).abs().max().item()}"


def test_every_fft_plan_matches_oracle(oracle):
    """Each compiled FFT plan (length N = T*E), forced on both axes, gives the
    same WFF2 result as the FP64 oracle on an image it covers."""
    plans = glsu.fft_plans()
    sig, lo, hi, st = 2.0, -0.6, 0.6, 0.3
    for p in plans:
        W = min(p["N"] - 6, 300)
        H = max(min(p["N"] - 6, 120), 16)
        say(f"[plan {p['id']}] T={p['T']} E={p['E']} N={p['N']} image {W}x{H} "
            f"exchange={p['exchange']}")
        rng = np.random.default_rng(p["id"])
        ph = 0.6 * np.arange(W)[None, :] + 0.25 * np.arange(H)[:, None] + rng.normal(0, 0.3, (H, W))
        f = np.exp(1j * ph).astype(np.complex64)
        ref = oracle.WFF2(W, H, sig, lo, hi, st)(f.astype(np.complex128))
        # rows use one wavefront per transform: narrow plans run on the column axis only
        px = p["id"] if p["T"] == 64 else -1
        w = glsu.WFT2(W, H, params=glsu.wff_params(sig, lo, hi, st), planx=px, plany=p["id"])
        out = w(torch.from_numpy(f).cuda()).cpu().numpy()
        rel = np.abs(out - ref).max() / np.abs(ref).max()
        say(f"   rel={rel:.2e}")
        assert rel < 1e-4, p


@pytest.mark.parametrize("W,H,T", [
    (818, 130, 64),   # 5 planes x 818 = 4090 columns: one transform per wavefront
    (820, 130, 16),   # 4100 columns: four narrow transforms per wavefront (192 points)
    (1000, 226, 64),  # exactly 256 points: no narrow plan is shorter
    (1000, 227, 16),  # one more: 320 narrow against 512
    (820, 290, 16),   # exactly 320 points
    (820, 291, 64),   # one more: 512 points, no narrow plan
    (33, 40, 64),     # a small image: rows over four wavefronts, columns in pairs
])
def test_default_column_plans_at_their_limits_match_oracle(oracle, W, H, T):
    """The default column plan follows the number of columns (planes x width)
    and the padded length; both sides of each limit against the oracle."""
    rng = np.random.default_rng(W + H)
    ph = 0.05 * np.arange(W)[None, :] - 0.08 * np.arange(H)[:, None] + rng.normal(0, 0.4, (H, W))
    f = np.exp(1j * ph).astype(np.complex64)
    ref = oracle.WFF2(W, H, 10.0, -0.2, 0.2, 0.1)(f.astype(np.complex128))
    w = glsu.WFT2(W, H, params=glsu.wff_params(10.0, -0.2, 0.2, 0.1))
    plans = {p["id"]: p for p in glsu.fft_plans()}
    assert plans[w.tuning()["plany"]]["T"] == T, w.tuning()
    out = w(torch.from_numpy(f).cuda()).cpu().numpy()
    rel = np.abs(out - ref).max() / np.abs(ref).max()
    rms, _ = wrapped_err(np.angle(out), np.angle(ref))
    say(f"   {W}x{H} {w.tuning()} rel={rel:.2e} phase rms={rms:.2e}")
    assert rel < 1e-4
    assert rms < 1e-4


@pytest.mark.parametrize("W,H,N", [
    (460, 98, 256),   # 2300 columns, 128 points needed: still one transform per wavefront
    (461, 98, 128),   # 2305 columns: four 128-point transforms per wavefront
    (600, 66, 128),   # 3000 columns, the middle of the range
    (461, 99, 256),   # 129 points needed: the 192-point plan's line is higher
])
def test_default_column_plan_of_short_images_matches_oracle(oracle, W, H, N):
    """The 128-point narrow plan pays from fewer columns than the longer ones;
    both sides of its line.  Bars as for the other defaults: FP32 transforms."""
    rng = np.random.default_rng(W + H)
    ph = 0.06 * np.arange(W)[None, :] + 0.05 * np.arange(H)[:, None] + rng.normal(0, 0.4, (H, W))
    f = np.exp(1j * ph).astype(np.complex64)
    ref = oracle.WFF2(W, H, 10.0, -0.2, 0.2, 0.1)(f.astype(np.complex128))
    w = glsu.WFT2(W, H, params=glsu.wff_params(10.0, -0.2, 0.2, 0.1))
    plans = {p["id"]: p for p in glsu.fft_plans()}
    assert plans[w.tuning()["plany"]]["N"] == N, w.tuning()
    out = w(torch.from_numpy(f).cuda()).cpu().numpy()
    rel = np.abs(out - ref).max() / np.abs(ref).max()
    rms, _ = wrapped_err(np.angle(out), np.angle(ref))
    say(f"   {W}x{H} {w.tuning()} rel={rel:.2e} phase rms={rms:.2e}")
    assert rel < 1e-4
    assert rms < 1e-4


@pytest.mark.parametrize("W,H,waves", [
    (200, 480, 2),    # 512 points, 1000 wavefronts: pairs
    (200, 483, 4),    # one row more: 768 points
    (200, 1000, 4),   # 1280 points
    (614, 482, 2),    # 3070 wavefronts
    (615, 482, 4),    # 3075
])
def test_default_column_workgroups_at_their_limits(W, H, waves):
    """Waves per workgroup of the column kernel by the plan's length and the
    wavefronts of the launch; the shape must not change the result."""
    rng = np.random.default_rng(W)
    f = np.exp(1j * rng.normal(0, 0.8, (H, W))).astype(np.complex64)
    params = glsu.wff_params(10.0, -0.2, 0.2, 0.1)
    w = glsu.WFT2(W, H, params=params)
    t = w.tuning()
    say(f"   {W}x{H} {t}")
    assert t["cols_waves"] == waves
    x = torch.from_numpy(f).cuda()
    o = glsu.WFT2(W, H, params=params, tuning=dict(t, cols_waves=6 - waves))
    assert o.tuning()["cols_waves"] == 6 - waves
    assert torch.equal(w(x), o(x))
