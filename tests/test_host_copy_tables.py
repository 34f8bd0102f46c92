"""The launch tables of the copy kernels, checked tile by tile on the CPU by a program built against the library
(tests/check_copy_tables.cpp): every tile is moved by exactly one workgroup, and no workgroup is launched without one."""
import os
import random
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "hccl_amd", "lib")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("tables") / "check_copy_tables")
    cmd = ["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT}/include", f"-I{ROOT}/hccl_amd/csrc",
           os.path.join(ROOT, "tests", "check_copy_tables.cpp"), "-o", exe, f"-L{LIB}", "-lhccl_amd", "-L/opt/rocm/lib", "-lamdhip64",
           f"-Wl,-rpath,{LIB}", "-Wl,-rpath,/opt/rocm/lib"]
    built = subprocess.run(cmd, capture_output=True, text=True)
    assert built.returncode == 0, built.stderr[-3000:]

    def run(*args):
        r = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return [int(x) for x in re.findall(r"\d+", r.stdout)]
    return run


def _matrix(kind, n):
    rng = random.Random(n)
    if kind == "equal":
        return [[70001] * n for _ in range(n)]
    if kind == "zipf":       # 2048 rows of 14336 bytes per rank, most of them for the first ranks
        w = [(j + 1) ** -1.2 for j in range(n)]
        return [[max(1, int(2048 * x / sum(w))) * 14336 for x in w] for _ in range(n)]
    if kind == "empty":      # four blocks of five empty, at the ends too
        return [[0 if (i * n + j) % 5 != 2 else rng.randint(1, 40000) for j in range(n)] for i in range(n)]
    m = [[rng.randint(1, 200) for _ in range(n)] for _ in range(n)]
    m[n - 1][0] = {"hot": 16 << 20, "huge": 2 << 30}[kind]
    return m


@pytest.mark.parametrize("kind", ["equal", "zipf", "hot", "huge", "empty"])
@pytest.mark.parametrize("n", [2, 3, 8, 15, 16, 48, 60, 63, 64])
def test_every_tile_of_an_alltoallv_is_found_once(check, n, kind):
    m = _matrix(kind, n)
    tiles, groups, size = check("blocks", n, *[c for row in m for c in row])
    payload = sum(c for row in m for c in row)
    live = sum(1 for row in m for c in row if c)
    # the grid: a block's tiles are its vectors, shifted by up to 63 of them, and one more for the bytes outside them
    assert tiles <= payload // 4096 + 2 * live
    # what is uploaded in front of the kernel
    assert groups <= 4096 and size <= 32 * live + 256 + 4 * (min(4096, 4 * live) + 1)


@pytest.mark.parametrize("max_groups,sources,most_launches", [
    (4096, ["65536:8x5000"], 1),                         # more sources than a launch has groups
    (4096, ["65536:8x6000"], 2),                         # more than its tables hold
    (4096, ["67108864:8", "4096:8x4090"], 1),            # one long source and many short ones
    (4096, ["100:2x4000", "1073741824:2"], 1),
    (4096, ["9000000:7x30", "70001:3x900", "1:2x50"], 1),
    (4096, ["8388608:8x7"], 1),
    (480, ["67108864:8", "1:8x63"], 1),                  # an AllGatherV in the kernel arguments
    (480, ["8388608:16x16"], 1),
    (480, ["33800:64x64"], 1),
    (480, ["1073745923:2", "1073741901:2"], 2),          # a source that begins in one launch and ends in the next
    (480, ["5368709120:3", "5:3"], 3),
])
def test_copies_to_several_places_launch_no_idle_workgroups(check, max_groups, sources, most_launches):
    """Every tile of every place exactly once; and as many workgroups as the sources have tiles at the worst alignment, times the
    launch's places, but for the last tiles of the batches and those in front of a source of 192 tiles or more."""
    tiles, workgroups, launches, _ = check("copies", max_groups, *sources)
    listed = [tuple(int(x) for x in (s if "x" in s else s + "x1").replace(":", "x").split("x")) for s in sources]
    most = max(places for _, places, _ in listed)
    own = sum(times * (size // 4096 + 2 + (7 if size // 4096 >= 190 else 0)) for size, _, times in listed)
    batches = own // 4000 + launches
    assert tiles <= workgroups <= most * (own + 8 * batches)
    assert launches <= most_launches


@pytest.mark.parametrize("gib,per_tile,ranks,fits", [(63, 4, 4, 1), (64, 4, 4, 0), (127, 4, 2, 1), (128, 4, 2, 0), (86, 4, 3, 0), (31, 2, 4, 1),
                                                     (32, 2, 4, 0), (15, 2, 8, 1), (16, 2, 8, 0), (22, 8, 16, 1), (33, 8, 16, 0)])
def test_a_wavefront_fold_stays_below_2_to_the_32_work_items(check, gib, per_tile, ranks, fits):
    """In place, 4 x 64 GiB or 2 x 128 GiB fit the memory, and the register kernel takes them."""
    assert fits == (gib * 2**20 // per_tile * 64 * ranks < 2**32)
    assert check("waves", gib * 2**20, per_tile, ranks) == [fits]
