"""The host loop of large read-outs (gpu-svo_amd/csrc/svo_ring.h), compiled
without a GPU against a thread that plays the device: every size around the
ring's 16 pieces of 512 KiB, with all helper threads, some, or none to be had,
and launches or waits that fail."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PIECE = 512 << 10


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("ring") / "readout_ring")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-pthread",
                    "-I", os.path.join(ROOT, "gpu-svo_amd", "csrc"),
                    os.path.join(ROOT, "tests", "readout_ring.cpp"), "-o", out], check=True)
    return out


def _run(program, *args):
    r = subprocess.run([program, *map(str, args)], check=True, capture_output=True, text=True,
                       timeout=60)
    return r.stdout.split()


@pytest.mark.parametrize("helpers", [0, 1, 3])
@pytest.mark.parametrize("delay_us", [0, 50])
@pytest.mark.parametrize("size", [1, PIECE, PIECE + 1, 2 * PIECE, 8 * PIECE, 16 * PIECE - 1,
                                  16 * PIECE, 16 * PIECE + 1, 18 * PIECE, 24 * PIECE + 7,
                                  80 * PIECE])
def test_bytes(program, size, delay_us, helpers):
    assert _run(program, size, helpers, delay_us, 0) == ["0", "same"]


@pytest.mark.parametrize("helpers", [0, 1, 3])
@pytest.mark.parametrize("fail_at", [1, 2, 10, 19, 40])
def test_failure_ends(program, helpers, fail_at):
    """The device's error comes back and every helper ends."""
    assert _run(program, 40 * PIECE, helpers, 0, fail_at)[0] == "-4"
