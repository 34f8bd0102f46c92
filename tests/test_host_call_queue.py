"""The queue of a rank's calls that wait for the other ranks' (csrc/host/call_queue.h): what it moves, holds and gives back, and
what is left of a call that could not be queued.  Host code only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "hccl_amd", "lib")


@pytest.fixture(scope="module")
def queue(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("queue") / "check_call_queue")
    subprocess.run(["g++", "-std=c++17", "-O2", f"-I{ROOT}/hccl_amd/csrc", os.path.join(ROOT, "tests", "check_call_queue.cpp"), "-o", exe],
                   check=True)
    return lambda n: [int(x) for x in subprocess.run([exe, str(n)], capture_output=True, text=True, check=True, timeout=60).stdout.split()]


@pytest.mark.parametrize("waiting", [1, 2, 63, 64, 65, 129, 1000, 20000])
def test_a_call_is_moved_a_bounded_number_of_times(queue, waiting):
    moves, most, left, wrong, out = queue(waiting)
    assert wrong == 0 and out >= waiting
    # in and out of the vector: 2; dropping the front moves no more calls than it drops: 1; growing the vector, which at
    # least doubles: 2
    assert moves <= 5 * out
    assert most <= 4 * max(64, waiting) and left <= 64


def test_a_call_that_could_not_be_queued_does_not_count(tmp_path):
    exe = str(tmp_path / "check_failed_push")
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT}/include", os.path.join(ROOT, "tests", "check_failed_push.cpp"), "-o", exe,
                    f"-L{LIB}", "-lhccl_amd", f"-Wl,-rpath,{LIB}"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", (run.returncode, run.stderr[-2000:])
