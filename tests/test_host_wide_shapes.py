"""Which shape a chain to one destination takes, on both sides of every limit of the rule, and which of them ask for LDS that they
do not use.  The rule is asked on the CPU by a program built against the library (tests/check_wide_shape.cpp)."""
import os
import subprocess

import pytest

from wide_shape_cases import CASES, CUS, SIZE, segment_lengths

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "hccl_amd", "lib")
MIB = 1 << 20


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("shape") / "check_wide_shape")
    cmd = ["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT}/include", f"-I{ROOT}/hccl_amd/csrc",
           os.path.join(ROOT, "tests", "check_wide_shape.cpp"), "-o", exe, f"-L{LIB}", "-lhccl_amd", "-L/opt/rocm/lib", "-lamdhip64",
           f"-Wl,-rpath,{LIB}", "-Wl,-rpath,/opt/rocm/lib"]
    built = subprocess.run(cmd, capture_output=True, text=True)
    assert built.returncode == 0, built.stderr[-3000:]

    def ask(esz, nsrc, off, *counts, hold=1, cus=CUS):
        run = subprocess.run([exe] + [str(a) for a in (cus, hold, esz, nsrc, off) + counts], capture_output=True, text=True, timeout=60)
        assert run.returncode == 0, run.stderr
        name, per_cu = run.stdout.split()
        return name, int(per_cu)
    return ask


@pytest.mark.parametrize("esz,nsrc", [(1, 5), (2, 8), (4, 5), (4, 8), (4, 64), (8, 16)])
def test_below_the_largest_no_launch_holds_lds(shape, esz, nsrc):
    """LDS that a fold does not use is LDS that kernels on other streams cannot have."""
    for mib in (1, 4, 7, 16, 25, 31, 33, 64, 72, 100, 127, 128, 143):
        for off in (0, esz):
            assert shape(esz, nsrc, off, mib * MIB // esz)[1] == 0


@pytest.mark.parametrize("esz", [1, 2, 4, 8])
def test_no_launch_holds_lds_when_told_not_to(shape, esz):
    for nsrc in (5, 8, 16, 64):
        for mib in (1, 16, 64, 128, 300, 1024, 4096):
            for off in (0, esz % 16):
                name, per_cu = shape(esz, nsrc, off, mib * MIB // esz, hold=0)
                assert per_cu == 0 and name != "large"


@pytest.mark.parametrize("dtype,op,nsrc,total,straddle,want", CASES)
def test_the_shape_of_what_runs_on_the_gpu(shape, dtype, op, nsrc, total, straddle, want):
    esz = SIZE[dtype]
    counts = segment_lengths(esz, total, straddle)
    assert sum(counts) * esz == total
    assert shape(esz, nsrc, esz if straddle else 0, *counts)[0] == want
