"""The tracers' compile-time variants and the step controller's limits.

- A kernel that integrates the coordinate time (ray records) and one that does not (frames of static
  turbulence, vacuum) trace the same rays: every pixel is the record's intensity rounded to float,
  bit for bit.
- The FP64 step at tolerances where its scaled error leaves the ordinary range (every step accepted at
  the largest growth, every step rejected, errors that overflow) against the oracle, bit for bit.
- The FP64 tracer at cameras whose steps pass near the pole and the horizon, likewise.
- The mixed vacuum step (its own form of the method) over spins, on and beside the spin axis, where the
  stage values of u decide the attempts: the FP64 tracer's fates, fewer attempts, and its escape angles
  to the far field's tolerance."""
import numpy as np
import pytest

import bhrt_amd as bh
from helpers import pixel_grid, setup, shot, tracer_for
from test_gpu_parity import assert_rays_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [bh.PREC_FP64, bh.PREC_MIXED])
@pytest.mark.parametrize("ini", ["c1_vacuum_256.ini", "c2_radio_1024.ini"])
def test_frames_equal_records(ini, prec):
    cfg = setup(shot(ini), W=83, H=41)
    t = tracer_for(cfg)
    try:
        for tol_t in (0.0, 1e-3):   # a bound on t asks for the coordinate time in frames too
            o = t.opts(precision=prec, tol_t=tol_t)
            img, _ = t.render(cfg["F"], o)
            rec = t.trace_tile(cfg["F"], 0, 0, 83, 41, o)
            assert np.array_equal(img.view(np.uint32), rec["I"].astype(np.float32).view(np.uint32)), tol_t
            assert (rec["y"][..., 5] != cfg["F"].t).all()
            frame, _ = t.render(cfg["F"], t.opts(precision=prec, tol_t=tol_t, engine=bh.ENGINE_FRAME))
            assert np.array_equal(img.view(np.uint32), frame.view(np.uint32)), tol_t
    finally:
        t.close()


@pytest.mark.parametrize("tol", [1e3, 1e-2, 1e-15, 1e-70, 1e-310, 0.0])
@pytest.mark.parametrize("ini", ["c1_vacuum_256.ini", "c2_radio_1024.ini"])
def test_extreme_tolerances(oracle_bhm, ini, tol):
    cfg = setup(shot(ini), W=256, H=256)
    cfg["S"].tol = cfg["OS"].tol = tol
    cfg["S"].max_steps = cfg["OS"].max_steps = 300
    t = tracer_for(cfg)
    try:
        gpu = t.trace_tile(cfg["F"], 120, 121, 17, 9)
        _, ref, _ = oracle_bhm.trace_pixels(cfg["OS"], cfg["OF"], *pixel_grid(17, 9, 120, 121))
        assert_rays_equal(gpu, ref, f"tol {tol}")
    finally:
        t.close()


@pytest.mark.parametrize("spin", [1e-6, 0.9999])
@pytest.mark.parametrize("incl", [0.02, 90.0, 179.9])
def test_pole_and_horizon(oracle_bhm, spin, incl):
    sets = f"bh.spin={spin!r};camera.incl={incl}"
    cfg = setup(shot("c2_radio_1024.ini"), sets, W=64, H=64)
    t = tracer_for(cfg)
    try:
        gpu = t.trace_tile(cfg["F"], 20, 21, 23, 22)
        _, ref, _ = oracle_bhm.trace_pixels(cfg["OS"], cfg["OF"], *pixel_grid(23, 22, 20, 21))
        assert_rays_equal(gpu, ref, sets)
    finally:
        t.close()


@pytest.mark.parametrize("spin", [1e-6, 0.5, 0.9999])
@pytest.mark.parametrize("cx", [0.0, 1e-3, 3.0])   # M from the axis to the image's centre column
def test_mixed_vacuum_step(spin, cx):
    sets = f"bh.spin={spin!r}"
    S = bh.build_scene(shot("c1_vacuum_256.ini"), sets)[0]
    F = bh.make_frame(S.a, 1000.0, 0.3, fov=16.0, off_x=cx, W=45, H=61)
    t = bh.Tracer(S)
    try:
        ref = t.trace_tile(F, 0, 0, 45, 61, t.opts())
        got = t.trace_tile(F, 0, 0, 45, 61, t.opts(precision=bh.PREC_MIXED))
        same = ref["fate"] == got["fate"]
        assert same.mean() > 0.998   # a ray on the critical curve may fall either way
        assert got["steps"].sum() < 0.6 * ref["steps"].sum()
        esc = same & (ref["fate"] == 1) & (ref["ncross"] <= 1)
        d = np.abs(np.cos(ref["th_inf"][esc]) - np.cos(got["th_inf"][esc]))
        assert esc.sum() > 500 and np.median(d) < 2e-5
    finally:
        t.close()
