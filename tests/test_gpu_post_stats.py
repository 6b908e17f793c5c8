"""The display statistics of a frame that fills the device path (65536 pixels and more, or 16384 and more
when it was blurred there) against the definition: the largest displayed intensity and the value of rank
floor(q (n - 1)) among those above 1e-5 of it, exactly; and the HUD over frames of every row shape."""
import numpy as np
import pytest

import bhrt_amd as bh
from helpers import setup, shot, tracer_for
from oracle_ctypes import Oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tracer():
    cfg = setup(shot("c1_vacuum_256.ini"), W=8, H=8)
    t = tracer_for(cfg)
    yield t
    t.close()


def stats(img, hide, q):
    v = img.reshape(-1, 4)
    with np.errstate(invalid="ignore"):
        d = ((v[:, 0] - v[:, 1]) - v[:, 2]) - v[:, 3]
        Y = v[:, 0] - np.float32(hide) * np.where(d < 0, np.float32(0), d)
        lum = Y[Y > 0]
        top = float(lum.max()) if lum.size else 0.0
        sig = np.sort(lum[lum.astype(np.float64) > top * 1e-5])
    return (float(sig[min(len(sig) - 1, int(q * (len(sig) - 1)))]) if len(sig) else 0.0), top


def frames():
    rng = np.random.default_rng(3)
    base = np.exp(rng.normal(-8, 4, (257, 263, 4))).astype(np.float32)
    base[..., 1:] *= np.float32(0.2)
    yield "log-normal", base
    yield "zero", np.zeros_like(base)
    yield "negative", -base
    one = np.zeros_like(base)
    one[100, 7, 0] = np.float32(1e-40)   # a denormal alone
    yield "one", one
    same = np.zeros_like(base)
    same[..., 0] = np.float32(0.75)
    yield "equal", same
    odd = base.copy()
    odd[3, 5, 0], odd[9, 9, 2] = np.nan, np.nan
    yield "nan", odd
    inf = base.copy()
    inf[0, 0, 0] = np.inf
    yield "inf", inf
    big = base.copy()
    big[-1, -1, 0] = np.float32(3e38)   # the threshold leaves this pixel alone
    yield "one above", big


@pytest.mark.parametrize("hide", [0.0, 0.3, 1.0])
def test_statistics(tracer, hide):
    for name, img in frames():
        for q in (0.0, 0.37, 0.995, 1.0):
            out, lp, lm = tracer.post_radio(img, 0.0, hide, q)
            assert np.array_equal(out.view(np.uint32), img.view(np.uint32))
            assert (lp, lm) == stats(img, hide, q), (name, q)


@pytest.mark.parametrize("size", [(127, 128), (128, 128), (129, 131), (1, 20000), (255, 256), (256, 256)])
def test_statistics_sizes(tracer, size):
    """Around the sizes at which the device path takes over, blurred and not."""
    img = np.abs(np.random.default_rng(5).normal(1, 1, (*size, 4))).astype(np.float32)
    for sigma in (0.0, 1.5, 9.0):
        out, lp, lm = tracer.post_radio(img, sigma, 0.3, 0.9)
        assert (lp, lm) == stats(out, 0.3, 0.9)


@pytest.mark.parametrize("W,H", [(1, 300), (3, 100), (255, 5), (256, 4), (257, 3), (1000, 2)])
def test_hud_row_shapes(tracer, W, H):
    """Workgroups that cover many rows, one row exactly, and parts of rows."""
    rng = np.random.default_rng(W)
    px = np.abs(rng.normal(0.3, 0.3, (H, W, 4))).astype(np.float32)
    atlas = rng.integers(0, 256, (20, 9, 7), dtype=np.uint8)
    rects = [(int(x), int(y), int(x + w), int(y + h), int(c), int(l)) for x, y, w, h, c, l in
             zip(rng.integers(-9, W + 9, 70), rng.integers(-9, H + 9, 70), rng.integers(-2, 40, 70),
                 rng.integers(-2, 40, 70), rng.integers(0, 1 << 32, 70), rng.integers(0, 3, 70))]
    glyphs = [(float(x), float(y), float(s), int(g), int(c)) for x, y, s, g, c in
              zip(rng.uniform(-20, W + 20, 600), rng.uniform(-20, H + 20, 600), rng.uniform(0.2, 4, 600),
                  rng.integers(0, 20, 600), rng.integers(0, 1 << 32, 600))]
    glyphs += [(3e9, 2.0, 1.0, 1, 0xFFFFFFFF), (-3e9, 2.0, 1.0, 1, 0xFFFFFFFF)]
    orc = Oracle("bhm")
    got = tracer.tonemap(px, rects=rects, glyphs=glyphs, atlas=atlas)
    want = orc.hud_draw(orc.tonemap_radio(px), glyphs, rects, atlas, max(1.5, H / 720.0))
    assert np.array_equal(got, want)
