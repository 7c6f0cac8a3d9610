"""Batched run of many uneven sequences (persistent launches, one graph per
frame step) against single-sequence handles with the same tuning: the
results must be bit-identical, frame by frame, also across repeated calls."""
import numpy as np
import pytest

from _util import say, wrapped_err

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import glsu  # noqa: E402

SIZES = [(96, 80), (256, 256), (300, 211), (512, 384), (130, 400), (256, 256), (77, 53)]
RRS = [1, 2, 1, 3, 1, 1, 2]


def _inputs(sizes, T, seed0=100):
    frames, phis = [], []
    for i, (W, H) in enumerate(sizes):
        amp0 = 2.0 + 3.0 * ((i * 0.37) % 1.0)
        frames.append(glsu.gen_frames(W, H, T, seed0 + i, amp0=amp0, noise=5.0 + 4.0 * i))
        phis.append(glsu.synth.phase(W, H, amp0, 0.05))
    return frames, phis


@pytest.mark.parametrize("graph", [True, False])
def test_batch_is_bitwise_equal_to_single_runs(graph):
    T = 5
    frames, phis = _inputs(SIZES, T)
    b = glsu.DPRABatch(phis, RRS)
    say(f"[batch] {len(SIZES)} sequences, info={b.info()}, graph={graph}")
    outs = b(frames, graph=graph)
    outs2 = b(frames, graph=graph)  # a second call continues from the state left
    for i, (W, H) in enumerate(SIZES):
        d = glsu.DPRA(phis[i], RRS[i], tuning=b.tuning(i))
        ref = d(frames[i]).cpu().numpy()
        ref2 = d(frames[i]).cpu().numpy()
        got, got2 = outs[i].cpu().numpy(), outs2[i].cpu().numpy()
        same = np.array_equal(got, ref) and np.array_equal(got2, ref2)
        say(f"   seq {i} {W}x{H} rr={RRS[i]} tuning={b.tuning(i)}: bitwise equal={same}")
        assert same, (i, np.abs(got - ref).max(), np.abs(got2 - ref2).max())
        p1, d1 = b.get_state(i)
        p2, d2 = d.get_state()
        assert np.array_equal(p1, p2) and np.array_equal(d1, d2)


def test_batch_with_explicit_tunings_and_oracle(oracle):
    sizes = [(200, 150), (128, 128)]
    T = 3
    frames, phis = _inputs(sizes, T, seed0=300)
    plans = {p["id"]: p for p in glsu.fft_plans()}
    narrow = [i for i, p in plans.items() if p["T"] != 64 and p["N"] >= 150 + 30][0]
    tunings = [dict(plany=narrow, cols_waves=2), dict(rows_waves=2)]
    b = glsu.DPRABatch(phis, 1, tunings=tunings)
    assert b.tuning(0)["plany"] == narrow and b.info()["classes"] == 2
    outs = b(frames)
    for i, (W, H) in enumerate(sizes):
        host = frames[i].cpu().numpy().astype(np.float64)
        ref = oracle.DPRA(phis[i]).run(host)
        for t in range(T):
            rms, mx = wrapped_err(outs[i][t].cpu().numpy(), ref[t])
            say(f"[batch vs oracle] seq {i} frame {t}: rms={rms:.2e} max={mx:.2e}")
            assert rms < 1e-3


def test_batch_long_transform_plans_are_bitwise_equal_to_single_runs():
    # plans with more than 24 elements per lane (64 x 36 = 2304 points) take
    # the kernels' read-ahead branches; forced here on small images so the
    # batched and single-frame kernels run them on the same inputs
    sizes = [(160, 120), (96, 200)]
    T = 3
    frames, phis = _inputs(sizes, T, seed0=700)
    plans = {p["id"]: p for p in glsu.fft_plans()}
    long_plan = [i for i, p in plans.items() if p["T"] == 64 and p["E"] > 24][0]
    tuning = dict(planx=long_plan, plany=long_plan, cols_waves=2, rows_waves=2)
    b = glsu.DPRABatch(phis, 1, tunings=[tuning, tuning])
    outs = b(frames)
    for i, (W, H) in enumerate(sizes):
        assert b.tuning(i)["plany"] == long_plan and b.tuning(i)["planx"] == long_plan
        ref = glsu.DPRA(phis[i], 1, tuning=b.tuning(i))(frames[i]).cpu().numpy()
        got = outs[i].cpu().numpy()
        say(f"[batch long plan {plans[long_plan]['N']}] seq {i} {W}x{H}: "
            f"bitwise equal={np.array_equal(got, ref)}")
        assert np.array_equal(got, ref), np.abs(got - ref).max()


def test_batch_uneven_workload_shape():
    """Sizes drawn from the uneven set (scaled down to 3 sizes, 12 sequences,
    3 frames): runs, and three sequences equal their single-handle runs."""
    rng = np.random.default_rng(5)
    sizes = [(int(s), int(s)) for s in rng.choice([256, 512, 768], 12)]
    frames, phis = _inputs(sizes, 3, seed0=500)
    b = glsu.DPRABatch(phis, 1)
    outs = b(frames, timed=True)
    say(f"[batch12] sizes={[s[0] for s in sizes]} classes={b.info()['classes']} "
        f"{b.last_ms:.2f} ms for 3 frames")
    for i in (0, 5, 11):
        ref = glsu.DPRA(phis[i], 1, tuning=b.tuning(i))(frames[i]).cpu().numpy()
        assert np.array_equal(outs[i].cpu().numpy(), ref)


@pytest.mark.parametrize("sizes,expect", [
    # (lanes per column transform, waves per workgroup) by image
    ([(256, 256)] * 2, [(64, 2)] * 2),                        # 2560 columns in the launch
    ([(256, 256)] * 16, [(16, 4)] * 16),                      # 20480 columns
    ([(96, 98)] * 5, [(16, 2)] * 5),                          # 2400 columns, 128 points
    ([(300, 400), (470, 400)], [(64, 4)] * 2),                # 1500 + 2350 columns
    ([(256, 256)] * 12 + [(256, 330)], [(64, 4)] * 13),       # 15360: not worth a class
    ([(256, 256)] * 13 + [(256, 330)], [(16, 4)] * 13 + [(64, 2)]),  # 16640, 4160 wavefronts
])
def test_batch_default_plans_follow_the_columns_of_the_launch(sizes, expect):
    """The columns of all images of a class run in one launch, so the default
    column plan and workgroup follow their sum, whatever the order of the
    list; results as on single handles with those tunings, bit for bit."""
    plans = {p["id"]: p for p in glsu.fft_plans()}
    for order in (1, -1):
        sz, ex = sizes[::order], expect[::order]
        frames, phis = _inputs(sz, 2, seed0=900)
        b = glsu.DPRABatch(phis, 1)
        got = [(plans[b.tuning(i)["plany"]]["T"], b.tuning(i)["cols_waves"])
               for i in range(len(sz))]
        say(f"[batch plans] {len(sz)} sequences {got} classes={b.info()['classes']}")
        assert got == ex
        outs = b(frames)
        for i in (0, len(sz) - 1):
            ref = glsu.DPRA(phis[i], 1, tuning=b.tuning(i))(frames[i])
            assert torch.equal(outs[i], ref)


def test_full_tunings_make_a_sequence_independent_of_the_others():
    """A sequence with the tuning of a handle of its own size gives that
    handle's results bit for bit, alone or beside any others."""
    sizes = [(256, 256)] * 16 + [(300, 211)]
    frames, phis = _inputs(sizes, 3, seed0=1100)
    own = []
    for i in (0, 16):
        d = glsu.DPRA(phis[i], 1)
        own.append((d.tuning(), d(frames[i])))
    tunings = [own[0][0]] * 16 + [own[1][0]]
    assert glsu.DPRABatch(phis, 1).tuning(0)["plany"] != own[0][0]["plany"]
    full = glsu.DPRABatch(phis, 1, tunings=tunings)(frames)
    pair = glsu.DPRABatch([phis[0], phis[16]], 1,
                          tunings=[own[0][0], own[1][0]])([frames[0], frames[16]])
    for k, i in enumerate((0, 16)):
        assert torch.equal(full[i], own[k][1]) and torch.equal(pair[k], own[k][1])
