"""Calls on a device that is nearly full: the normalising flux and the display statistics keep working where their
faster paths' buffers cannot be had, with the results of those paths, and the flux gives a large buffer back."""
import numpy as np
import pytest
import torch

import bhrt_amd as bh
from helpers import setup, shot, tracer_for

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def fill(left, needed):
    """Takes the device's free memory but for about `left` bytes, too few for a buffer of `needed`."""
    hogs = []
    for _ in range(16):
        extra = torch.cuda.mem_get_info()[0] - left
        if extra < 16 * MIB:
            break
        hogs.append(torch.empty(extra, dtype=torch.uint8, device="cuda"))
    assert torch.cuda.mem_get_info()[0] < needed
    return hogs


def test_flux_without_room_for_its_samples():
    r = setup(shot("c2_radio_1024.ini"), W=64, H=64)
    t = tracer_for(r)
    n = 4096                # 1 GiB of samples
    try:
        t.radio_flux(r["F"], 512, 1e-20)
        before = torch.cuda.mem_get_info()[0]
        want = t.radio_flux(r["F"], n, 1e-20)
        assert torch.cuda.mem_get_info()[0] > before - 512 * MIB   # the samples were given back
        t.render(r["F"], t.opts(engine=bh.ENGINE_FRAME, spp=2, jitter=1))
        hogs = fill(700 * MIB, 2 * n * n * 32)
        try:
            got = t.radio_flux(r["F"], n, 1e-20)
            small = t.radio_flux(r["F"], 64, 1e-20)
        finally:
            del hogs
            torch.cuda.empty_cache()
        assert got == want and small > 0.0   # the same blocks and order of additions
        assert t.radio_flux(r["F"], n, 1e-20) == want
    finally:
        t.close()


def test_statistics_without_room_for_the_frame():
    r = setup(shot("c2_radio_1024.ini"), W=64, H=64)
    t = tracer_for(r)
    W, H = 8192, 6144   # 768 MiB
    rng = np.random.default_rng(1)
    img = np.zeros((H, W, 4), dtype=np.float32)
    img[..., 0] = rng.random((H, W), dtype=np.float32) ** 8
    img[:, ::5, 0] = 0.0
    try:
        want = t.post_radio(img)[1:]
    finally:
        t.close()
    t = tracer_for(r)   # holds none of the buffers
    try:
        hogs = fill(600 * MIB, img.nbytes)
        try:
            got = t.post_radio(img)[1:]
        finally:
            del hogs
            torch.cuda.empty_cache()
        assert got == want and want[1] == img[..., 0].max()
        assert t.post_radio(img)[1:] == want
    finally:
        t.close()
