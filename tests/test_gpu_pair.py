"""Radio launches of few rays, which integrate in one wave and evaluate the flow in another, against the frame
kernel, which does both in turn: the same records bit for bit. Sizes from one ray to several generations of
rays per workgroup; static, time-sliced and sheared turbulence; rays that become opaque on the way (they run
ahead of their samples and are taken back) and rays that end at the step limit, at either side of an interval
of 64 attempts. Frames of several sizes and spins in one launch against a launch configuration of its own,
which keeps the plain kernel."""
import numpy as np
import pytest

import bhrt_amd as bh
from helpers import shot
from test_gpu_batch import assert_records_same

pytestmark = pytest.mark.gpu

N0 = 291464.0


def tracer(turb, n0=N0, max_steps=0):
    S, k2, (l0, dl), _, _ = bh.build_scene(shot("c2_radio_1024.ini"), "")
    S.n0 = n0
    if max_steps:
        S.max_steps = max_steps
    kw = dict(turb_model=bh.TURB_SHEARED, ts_dims=(96, 32, 12, 6))
    if turb != "sheared":
        nt = 8 if turb == "slices" else 1
        kw = dict(grid=bh.turbulence(32, nt, 60.0, 0.3, 5.0, 30.0, 10.0, 3), turb_half=60.0, turb_t0=-1080.0, turb_dt=20.0)
    return S, bh.Tracer(S, k2=k2, k2_l0=l0, k2_dl=dl, **kw)


def compare(t, F, x0, y0, w, h, prec, what):
    got = t.trace_tile(F, x0, y0, w, h, t.opts(precision=prec, jitter=1))
    want = t.trace_tile(F, x0, y0, w, h, t.opts(precision=prec, jitter=1, engine=bh.ENGINE_FRAME))
    assert_records_same(got, want, what)
    return got


@pytest.mark.parametrize("prec", [bh.PREC_FP64, bh.PREC_MIXED])
@pytest.mark.parametrize("turb", ["grid", "slices", "sheared"])
def test_records(prec, turb):
    S, t = tracer(turb)
    try:
        F = bh.make_frame(S.a, 1000.0, 0.3, fov=24.0, W=256, H=200)
        for x0, y0, w, h in ((130, 60, 1, 1), (64, 64, 8, 8), (101, 37, 65, 9), (0, 0, 256, 200)):
            q = compare(t, F, x0, y0, w, h, prec, f"{turb} {w}x{h}")
        assert (q["fate"] == 1).any() and (q["fate"] == -1).any() and (q["flow_steps"] > 64).any()
    finally:
        t.close()


@pytest.mark.parametrize("prec", [bh.PREC_FP64, bh.PREC_MIXED])
def test_opaque_rays(prec):
    S, t = tracer("grid", n0=3e3 * N0)
    try:
        F = bh.make_frame(S.a, 1000.0, 1.2, fov=30.0, W=96, H=72)
        q = compare(t, F, 0, 0, 96, 72, prec, "opaque")
        opaque = (q["trans"] < 1e-5) & (q["fate"] == -1)
        assert opaque.mean() > 0.05 and len(np.unique(q["steps"][opaque] % 64)) > 32
    finally:
        t.close()


@pytest.mark.parametrize("prec", [bh.PREC_FP64, bh.PREC_MIXED])
@pytest.mark.parametrize("max_steps", [1, 63, 64, 65, 130])
def test_step_limit(prec, max_steps):
    S, t = tracer("grid", max_steps=max_steps)
    try:
        F = bh.make_frame(S.a, 1000.0, 0.3, fov=30.0, W=64, H=48)
        q = compare(t, F, 0, 0, 64, 48, prec, f"limit {max_steps}")
        assert (q["steps"] <= max_steps).all() and (q["steps"] == max_steps).any()
    finally:
        t.close()


@pytest.mark.parametrize("prec", [bh.PREC_FP64, bh.PREC_MIXED])
def test_batch_of_frames(prec):
    S, t = tracer("slices")
    try:
        frames = []
        for i, (spin, w, h) in enumerate([(0.0, 40, 24), (0.94, 1, 1), (0.998, 97, 63)]):
            Si = bh.build_scene(shot("c2_radio_1024.ini"), f"bh.spin={spin}")[0]
            Si.n0 = N0 * (1 + 2e3 * (i == 2))   # the last frame optically thick
            frames.append((Si, bh.make_frame(Si.a, 1000.0, 0.5, fov=30.0, W=w, H=h)))
        o = t.opts(precision=prec)
        got, st = t.trace_batch(frames, o)
        want, sw = t.trace_batch(frames, o, block=64, grid_per_cu=2, interval=16, waves=3)
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert (st.step_attempts, st.steps_accepted, st.flow_steps, st.step_limited) == \
               (sw.step_attempts, sw.steps_accepted, sw.flow_steps, sw.step_limited)
    finally:
        t.close()
