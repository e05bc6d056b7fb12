"""The split-K scratch of settling plans, on the CPU: tests/plan_check builds the library's own host planner and looks
at every step's problems."""
import os
import subprocess

import pytest

from predicitivecoding_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def plan_check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan_check") / "plan_check")
    # the phase kernels' launchers are never called here, so their units are not built
    res = subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *build.HIPCC_FLAGS, "-O1", "-x", "hip",
                          os.path.join(HERE, "plan_check", "plan_check.hip"), "-o", out,
                          "-Wl,--unresolved-symbols=ignore-all"], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
    return out


def run(exe, *args):
    res = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
    return res.returncode, res.stdout


@pytest.mark.parametrize("dtype,rows,sizes", [
    (0, 1732, [768] * 5), (1, 319, [2048] * 6), (2, 319, [2048] * 6), (0, 700, [3584] * 3)])
def test_one_row_problems_near_the_scratch_end_stay_inside(plan_check, dtype, rows, sizes):
    """Full phases that do not split, with fewer than half as many tiles as CUs once layers are down to one row."""
    rc, out = run(plan_check, dtype, rows, *sizes)
    assert rc == 0 and "1 with shared rows" in out, out


@pytest.mark.parametrize("seed", [1, 2])
def test_random_plans_stay_inside_their_scratch(plan_check, seed):
    rc, out = run(plan_check, seed, 20000)
    assert rc == 0, out[-2000:]
    assert int(out.split("accepted, ")[1].split()[0]) > 10000, out   # plans with shared rows are among them


@pytest.mark.parametrize("rows,sizes,tile", [
    (1024, [1024] * 4 + [256], 128),     # a 128 x 128 tile on every CU, four of 64 x 64
    (1476, [836] * 4, 64),               # 252 tiles, but 33 on some XCDs of 32 CUs
    (1293, [1024] * 4, 64),              # 264: two rounds against four
    (892, [1408] * 4, 128),              # 231 of 256 CUs, one round against four
    (500, [1024] * 7, 64),               # one against three
    (1600, [1024] * 5, 128),             # two rounds against seven
    (892, [700] * 8, 64),                # a mean K of 700
    (686, [107, 520, 95, 74, 84, 1724, 1281, 1494, 233], 64),   # unlike layers
    (3000, [512] * 12, 128),             # two and more 128 x 128 tiles on every CU, whatever K
])
def test_fp32_tile_choice(plan_check, rows, sizes, tile):
    _, out = run(plan_check, 0, rows, *sizes)
    assert out.startswith(f"tile {tile}\n"), out
