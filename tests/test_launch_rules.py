"""The rules that shape a persistent launch (csrc/launch.h), compiled with the host compiler: which radio launches
integrate and evaluate in two waves, by the number of rays, how many of them reach the emitting region, and
whether the flow is opaque; the share of a region's rays that pass within a radius, against the area; the
defaults at either side of their lines; and which launches a tuned configuration holds for."""
import math
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FP64, MIXED = 0, 1


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "rules")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-o", exe,
                    os.path.join(HERE, "launch_rules", "rules.cpp")], check=True)

    def ask(*lines):
        out = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True).stdout
        return [float(x) for x in out.split()]
    return ask


@pytest.mark.parametrize("prec,w,reach,opaque,want", [
    (FP64, 0.1, 0.1, 0, 1), (FP64, 10.0, 10.0, 0, 1), (FP64, 10.1, 10.1, 0, 0), (FP64, 9.0, 9.0, 1, 1),
    (MIXED, 0.1, 0.1, 1, 1), (MIXED, 12.0, 12.0, 1, 1), (MIXED, 12.3, 12.3, 1, 0),   # an opaque flow, all rays in it
    (MIXED, 25.0, 11.0, 1, 1), (MIXED, 25.0, 15.0, 1, 0),                            # few of them in it
    (MIXED, 22.6, 22.6, 0, 1), (MIXED, 25.0, 25.0, 0, 0),                            # a thin one, all rays in it
    (MIXED, 39.8, 17.0, 0, 1), (MIXED, 40.1, 1.0, 0, 0),
])
def test_pairs(rules, prec, w, reach, opaque, want):
    assert rules(f"{prec} 1 {w} {reach} {opaque}") == [want]
    assert rules(f"{prec} 0 {w} {reach} {opaque}") == [0]   # vacuum: nothing to evaluate


@pytest.mark.parametrize("r,fov,w,h,want", [
    (10.0, 40.0, 1024, 1024, math.pi / 16), (100.0, 40.0, 640, 480, 1.0), (0.0, 40.0, 64, 64, 0.0),
    (15.0, 40.0, 512, 256, None),
])
def test_share(rules, r, fov, w, h, want):
    pix = fov / w / 1000.0
    got, = rules(f"share {r} 1000 0 0 {pix!r} {w} {h} 0 0 {w} {h}")
    if want is None:   # a frame twice as wide as high: the disc is cut at |y| = 10
        y = fov * h / w / 2
        want = (2 * (y * math.sqrt(r * r - y * y) + r * r * math.asin(y / r))) / (fov * fov * h / w)
    assert abs(got - want) <= 0.05   # 256 sample points: the edge passes through some 40 of them


def test_share_off_centre(rules):
    pix = 40.0 / 1000 / 1000.0
    # a frame beside the disc, one inside it, a region of a frame that holds the disc, one that misses it
    assert rules(f"share 10 1000 0.05 0 {pix!r} 1000 1000 0 0 1000 1000", f"share 30 1000 0 0 {pix!r} 1000 1000 0 0 1000 1000",
                 f"share 10 1000 0 0 {pix!r} 1000 1000 400 400 200 200",
                 f"share 10 1000 0 0 {pix!r} 1000 1000 0 0 200 200") == [0.0, 1.0, 1.0, 0.0]


@pytest.mark.parametrize("load,want", [
    ("0 1 0.1 0.1 0", [64, 4, 1, 1]), ("0 1 10 10 0", [64, 4, 3, 1]), ("0 1 10.1 10.1 0", [64, 8, 3, 0]),
    ("0 1 20.1 20.1 0", [256, 3, 3, 0]), ("0 2 64 64 0", [256, 3, 1, 0]),
    ("0 0 2.9 2.9 0", [64, 3, 1, 0]), ("0 0 6.9 6.9 0", [64, 4, 3, 0]), ("0 0 7.1 7.1 0", [64, 8, 3, 0]),
    ("1 1 0.1 0.1 0", [64, 4, 3, 1]), ("1 2 39.9 17 0", [64, 4, 3, 1]), ("1 1 20 20 1", [256, 2, 3, 0]),
    ("1 1 48.1 9 0", [256, 3, 3, 0]), ("1 0 8 8 0", [256, 1, 3, 0]), ("1 0 8.1 8.1 0", [256, 3, 3, 0]),
])
def test_defaults(rules, load, want):
    assert rules(f"defaults {load}") == want


SMALL, LARGE, VACUUM = "{p} 1 1 1 0", "{p} 1 64 30 0", "{p} 0 64 64 0"


@pytest.mark.parametrize("p", [FP64, MIXED])
def test_tuned_holds_for_launches_like_it(rules, p):
    small, large, vacuum = (x.format(p=p) for x in (SMALL, LARGE, VACUUM))
    # tuned on many rays: holds for as many and more, not for few, which keep the two waves
    assert rules(f"tuned {large} {large} 128 8 32") == [128, 8, 32, 0]
    assert rules(f"tuned {large} {p} 1 300 200 0 128 8 32") == [128, 8, 32, 0]
    assert rules(f"tuned {large} {small} 128 8 32") == [64, 4, 64, 1]
    # tuned on few rays: the shape of a launch that waits for its longest ray is not forced on many
    assert rules(f"tuned {small} {small} 64 4 16") == [64, 4, 16, 1]
    assert rules(f"tuned {small} {small} 64 1 64") == [64, 1, 64, 0]
    assert rules(f"tuned {small} {large} 64 1 64")[:2] != [64, 1]
    # tuned with a flow, used without one
    assert rules(f"tuned {large} {vacuum} 128 8 32")[0] == 256


@pytest.mark.parametrize("w,per_cu,order", [(2.9, 3, 1), (4.0, 3, 1), (4.1, 4, 3), (5.0, 4, 3)])
def test_fp64_sorts_what_it_does_not_hold(rules, w, per_cu, order):
    """Beyond one wave of rays per SIMD the longest rays go first."""
    assert rules(f"defaults 0 0 {w} {w} 0") == [64, per_cu, order, 0]
    assert rules(f"defaults 0 1 {w} {w} 0") == [64, 4, order, 1]
