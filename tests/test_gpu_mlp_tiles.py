"""Surrogate gradient and inference at the edges of their work layout: a workgroup whose second tile is
empty, an odd number of tiles, a last tile of one sample, and more tiles than persistent workgroups.
Both against the double-precision oracle (oracle/mlp_ref.py), with the bounds of split-BF16 products:
operands carry 16 bits (2^-16 relative error each), and sums of at most 64 terms of mixed sign stay
within a few times that, 1e-4 of the largest element."""
import numpy as np
import pytest

import bhrt_amd as bh  # noqa: F401
import mlp_ref as M
from helpers import setup, shot, tracer_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tracer():
    t = tracer_for(setup(shot("c2_radio_1024.ini")))
    yield t
    t.close()


def params(seed):
    c, h = M.default_input_norm()
    norm = np.concatenate([c, h, [-6.0, -30.0, 8.0, 15.0]]).astype(np.float32)
    return (np.random.default_rng(seed).normal(size=M.NPARAM) * 0.25).astype(np.float32), norm


@pytest.mark.parametrize("n", [16, 32, 48, 8208])
def test_gradient_tile_edges(tracer, n):
    p, norm = params(n)
    rng = np.random.default_rng(n + 1)
    xn = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    tr = (rng.normal(size=(n, 2)) * norm[8:10] + norm[6:8]).astype(np.float32)
    w = rng.uniform(0.5, 3.0, n).astype(np.float32)
    loss, g = tracer.mlp_grad(p, norm, xn, tr, w)
    loss_ref, g_ref = M.loss_and_grad(p.astype(np.float64), norm, xn, tr, w)
    assert abs(loss - loss_ref) <= 1e-4 * loss_ref
    cuts = [M.OFF_W1, M.OFF_B1, M.OFF_W2, M.OFF_B2, M.OFF_W3, M.OFF_B3, M.OFF_W4, M.OFF_B4, M.NPARAM]
    for a, b in zip(cuts, cuts[1:]):
        assert np.abs(g[a:b] - g_ref[a:b]).max() <= 1e-4 * np.abs(g_ref[a:b]).max(), (a, b)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 2048 * 16 + 1])
def test_inference_tile_edges(tracer, n):
    p, norm = params(7)
    tracer.mlp_set(p, norm)
    rng = np.random.default_rng(n)
    x = np.column_stack([rng.uniform(-4, 6, n), np.exp(rng.uniform(np.log(0.5), np.log(100), n)),
                         rng.uniform(0.01, np.pi - 0.01, n)]).astype(np.float32)
    got = tracer.mlp_infer(x[:, 0], x[:, 1], x[:, 2])
    x = x.astype(np.float64)
    y, _ = M.forward(p, M.normalise_inputs(x[:, 0], x[:, 1], x[:, 2], norm))
    assert (np.abs(got - (y * norm[8:10] + norm[6:8])) / norm[8:10]).max() < 1e-4
