"""The waits for the pinned ring (gpu-svo_amd/csrc/svo_ring.h), compiled
without a GPU: a device that answers late does not cost its waiters a core,
and one that ends without an answer ends the wait."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("waits") / "ring_waits")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-pthread",
                    "-I", os.path.join(ROOT, "gpu-svo_amd", "csrc"),
                    os.path.join(ROOT, "tests", "ring_waits.cpp"), "-o", out], check=True)
    return out


def _run(program, mode, ms):
    r = subprocess.run([program, mode, str(ms)], check=True, capture_output=True, text=True,
                       timeout=60)
    ok, cpu = r.stdout.split()
    return int(ok), float(cpu)


@pytest.mark.parametrize("mode,threads", [("lookup", 1), ("read", 4)])
def test_late_answers_cost_no_core(program, mode, threads):
    """400 ms late.  Each thread spins for 0.2 ms, then sleeps for an eighth of
    the time waited, 1 ms at most: 460 wake-ups (40 up to 8 ms, where the
    millisecond holds, 400 after), of a few us each."""
    ok, cpu = _run(program, mode, 400)
    assert ok == 1 and cpu < 40.0 * threads, cpu


@pytest.mark.parametrize("ms", [0, 1, 50])
def test_ends(program, ms):
    assert _run(program, "dead", ms)[0] == 0
    assert _run(program, "last", ms)[0] == 1
    assert _run(program, "lookup", ms)[0] == 1
