"""One step of the mixed vacuum tracer's form of Dormand-Prince 5(4) (dp54_n) against one step of the FP64
tracer's, from the same state with the same step size (2 % of the radial scale, where the second-order terms are
4e-4 of r): every component of the state. Both round in FP64; sums of at most nine terms and quotients by
Delta sin^2 theta (at least 0.1 of its terms here) stay within 1e-13 of the components' scales."""
import numpy as np
import pytest

import bhrt_amd as bh
from helpers import shot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spin", [1e-6, 0.5, 0.94, 0.9999])
@pytest.mark.parametrize("r,incl", [(6.0, 1.0), (8.0, 0.5), (20.0, 1.5), (200.0, 2.6)])
def test_one_step(spin, r, incl):
    S = bh.build_scene(shot("c1_vacuum_256.ini"), f"bh.spin={spin!r}")[0]
    S.max_steps = 1
    S.tol = 1e-5
    F = bh.make_frame(S.a, r, incl, fov=r, W=64, H=64)
    t = bh.Tracer(S)
    try:
        a = t.trace_tile(F, 0, 0, 64, 64, t.opts())
        b = t.trace_tile(F, 0, 0, 64, 64, t.opts(precision=bh.PREC_MIXED))
        both = (a["accepted"] == 1) & (b["accepted"] == 1)
        assert both.mean() > 0.99
        ya, yb = a["y"][both], b["y"][both]
        assert (np.abs(ya[:, 0] - r) > 1e-3 * r).mean() > 0.9   # the rays moved
        scale = np.stack([ya[:, 0], ya[:, 0] ** 2, np.ones(len(ya)), ya[:, 0], 1.0 + np.abs(ya[:, 4]),
                          ya[:, 0] + np.abs(ya[:, 5])], axis=1)
        assert (np.abs(ya - yb) / scale).max() <= 1e-13
        assert (ya != yb).any()   # two forms, not one
    finally:
        t.close()
