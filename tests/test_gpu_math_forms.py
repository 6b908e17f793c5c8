"""The FP64 tracer's own forms of the quotient, the root, the step controller's factor and the swept angle on the
device, bit for bit against the operations they stand for (IEEE division and root, the oracle's x^-0.2 and atan2),
over the domains they state: operands and results within 2^+-900, zeros, infinities and NaN where a form takes
them; errors from 0 to infinity, at the controller's limits and across them; directions of every octant, the axes
and vectors that are a few ulp off unit length."""
import numpy as np
import pytest

import bhrt_amd as bh

pytestmark = pytest.mark.gpu

N = 1_000_000


def same(got, want):
    g, w = got.view(np.int64), want.view(np.int64)
    bad = (g != w) & ~(np.isnan(got) & np.isnan(want))
    assert not bad.any(), (bad.sum(), np.flatnonzero(bad)[:5], got[bad][:5], want[bad][:5])


def significands(rng, n):
    """Random ones, and those next to 1, to 2 and to a power of two plus or minus a few ulp."""
    m = rng.uniform(1.0, 2.0, n)
    k = rng.integers(0, 8, n // 4)
    m[: n // 8] = 1.0 + k[: n // 8] * 2.0**-52
    m[n // 8: n // 4] = 2.0 - (1 + k[: n // 4 - n // 8]) * 2.0**-52
    return rng.permutation(m)


def test_quotient():
    rng = np.random.default_rng(11)
    for e in (0, 30, 440):
        x = significands(rng, N) * 2.0 ** rng.integers(-e, e + 1, N) * rng.choice([-1.0, 1.0], N)
        y = significands(rng, N) * 2.0 ** rng.integers(-e, e + 1, N)
        same(bh.math_eval("quot", x, y), x / y)
    edge = np.array([0.0, 1.0, 3.0, 1e200, np.inf, np.nan])
    x, y = (v.ravel() for v in np.meshgrid(np.concatenate([edge, -edge]), edge))
    with np.errstate(all="ignore"):
        same(bh.math_eval("quot", x, y), x / y)


def test_root():
    rng = np.random.default_rng(12)
    for e in (0, 1, 60, 900):
        x = significands(rng, N) * 2.0 ** rng.integers(-e, e + 1, N)
        same(bh.math_eval("root", x), np.sqrt(x))
    squares = np.arange(1.0, 100001.0) ** 2
    for x in (squares, np.nextafter(squares, 0.0), np.nextafter(squares, np.inf), np.zeros(1)):
        same(bh.math_eval("root", x), np.sqrt(x))


def test_step_factor(oracle_bhm):
    rng = np.random.default_rng(13)
    err = np.concatenate([np.exp(rng.uniform(np.log(1e-7), np.log(1e7), 2 * N)), 10.0 ** rng.uniform(-300, 300, N // 4),
                          np.exp(rng.uniform(np.log(1.8e-4), np.log(1.9e-4), N // 4)),   # the factor reaches 5 ...
                          np.exp(rng.uniform(np.log(1.84e3), np.log(1.85e3), N // 4)),   # ... and 0.2
                          [0.0, 1e-310, 1e-6, 1.0, 1e6, 1e300, np.inf]])
    want = np.minimum(5.0, np.maximum(0.2, 0.9 * oracle_bhm.math_eval("pow_m02", np.clip(err, 1e-30, 1e300))))
    same(bh.math_eval("step_factor", err), want)


def test_angle(oracle_bhm):
    rng = np.random.default_rng(14)
    a = np.concatenate([rng.uniform(0.0, np.pi, N), np.exp(rng.uniform(-30.0, 0.0, N // 2)),
                        np.pi - np.exp(rng.uniform(-30.0, 0.0, N // 2)), np.arange(5) * np.pi / 4])
    k = 1.0 + rng.integers(-8, 9, a.size) * 2.0**-52
    y, x = np.abs(np.sin(a)) * k, np.cos(a) * k
    y = np.concatenate([y, [0.0, 0.0, 1.0, 0.5**0.5, 0.5**0.5]])
    x = np.concatenate([x, [1.0, -1.0, 0.0, 0.5**0.5, -(0.5**0.5)]])
    same(bh.math_eval("angle", y, x), oracle_bhm.math_eval("atan2", y, x))
