"""The threaded copy to pageable memory (csrc/transfer.h) on a stream driven by the test: its threads sleep while
the stream is still busy with what was queued before the copy, there are no more of them than the process has
cores (none for one or two), every byte arrives and none beyond, and a failing copy is reported."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CORES = len(os.sched_getaffinity(0))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("transfer") / "transfer")
    src = os.path.join(HERE, "transfer")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-pthread", "-I", src, "-o", out, os.path.join(src, "transfer.cpp")],
                   check=True)
    return out


@pytest.mark.parametrize("cpus", [0, 1, 2, 3, 5])
def test_transfer(exe, cpus):
    if cpus > CORES:
        pytest.skip(f"{CORES} cores")
    out = subprocess.run([exe, str(cpus)], capture_output=True, text=True, timeout=60, check=True).stdout.split()
    threads, busy, right, reported = int(out[0]), float(out[1]), int(out[2]), int(out[3])
    cores = cpus or CORES
    assert right and reported
    assert threads <= (1 if cores <= 2 else min(cores, 8))
    # 0.4 s of other work on the stream: the copy itself takes a few ms on each of its threads
    assert busy < 0.2
