"""Optically thick flows on the launches that integrate in one wave and evaluate in another: a ray whose sample
made it opaque stops within two attempts, so the launch is not slower than the plain engine on the same rays
(launch times in turn, medians of nine; 1.25 allows for their spread of some 10 %)."""
import numpy as np
import pytest

import bhrt_amd as bh
from helpers import shot

pytestmark = pytest.mark.gpu

N0 = 291464.0


@pytest.mark.parametrize("prec,size", [(bh.PREC_MIXED, 448), (bh.PREC_MIXED, 640), (bh.PREC_FP64, 256)])
def test_thick_flow_time(prec, size):
    S, k2, (l0, dl), _, _ = bh.build_scene(shot("c2_radio_1024.ini"), "")
    S.n0 = 3000 * N0
    t = bh.Tracer(S, k2=k2, k2_l0=l0, k2_dl=dl, grid=bh.turbulence(32, 1, 60.0, 0.3, 5.0, 30.0, 10.0, 3), turb_half=60.0)
    try:
        frames = [(S, bh.make_frame(S.a, 1000.0, 1.2, fov=30.0, W=size, H=size))]
        o = t.opts(precision=prec)
        ms = {"default": [], "plain": []}
        for i in range(10):
            for name, cfg in (("default", {}), ("plain", dict(block=256, grid_per_cu=2, interval=48, waves=3))):
                _, st = t.trace_batch(frames, o, resident=True, **cfg)
                if i:
                    ms[name].append(st.ms_kernel)
        a, b = np.median(ms["default"]), np.median(ms["plain"])
        print(f"default {a:.3f} ms, plain {b:.3f} ms")
        assert a <= 1.25 * b
    finally:
        t.close()


@pytest.mark.parametrize("interval", [1, 2, 3, 5, 64])
@pytest.mark.parametrize("prec,far_fp32,full_flow", [(bh.PREC_FP64, 0, 0), (bh.PREC_MIXED, 0, 0), (bh.PREC_MIXED, 1, 0),
                                                     (bh.PREC_MIXED, 1, 1)])
def test_opaque_rays_pixels_and_statistics(prec, far_fp32, full_flow, interval):
    """Rays that turn opaque in any attempt of an interval, its last two among them, against the plain engine: the
    pixels and every statistic. The shape 64 / 4 / waves 3 is the two waves', with any interval."""
    S, k2, (l0, dl), _, _ = bh.build_scene(shot("c2_radio_1024.ini"), "")
    S.n0 = 1000 * N0
    t = bh.Tracer(S, k2=k2, k2_l0=l0, k2_dl=dl, grid=bh.turbulence(32, 1, 60.0, 0.3, 5.0, 30.0, 10.0, 3), turb_half=60.0)
    try:
        frames = [(S, bh.make_frame(S.a, 1000.0, 1.0, fov=60.0, W=75, H=52)),
                  (S, bh.make_frame(S.a, 1000.0, 0.3, fov=100.0, W=33, H=21))]
        o = t.opts(precision=prec, far_fp32=far_fp32, full_flow=full_flow)
        got, sg = t.trace_batch(frames, o, block=64, grid_per_cu=4, interval=interval, waves=3)
        want, sw = t.trace_batch(frames, o, block=128, grid_per_cu=2, interval=16, waves=3)
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        for f in ("samples", "step_limited", "step_attempts", "steps_accepted", "flow_steps", "fp64_steps"):
            assert getattr(sg, f) == getattr(sw, f), f
        if far_fp32:
            assert sg.fp64_steps < sg.step_attempts
    finally:
        t.close()
