"""CPU: every device address and every store of the whole-grid fused step, enumerated by
a C++ program (tests/march_check.cpp) from the kernel's own geometry functions and the
library's launch geometry: reads inside the arrays, each cell and each memory variable
stored exactly once."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
LIB = os.path.join(ROOT, "ela3d_amd", "libela3d.so")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if not os.path.exists(HIPCC) or not os.path.exists(LIB):
        pytest.skip("needs hipcc and the built library")
    exe = str(tmp_path_factory.mktemp("mc") / "march_check")
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    os.path.join(ROOT, "tests", "march_check.cpp"), f"-I{os.path.join(ROOT, 'ela3d_amd', 'csrc')}",
                    f"-I{os.path.join(ROOT, 'include')}", f"-L{os.path.dirname(LIB)}", "-lela3d",
                    f"-Wl,-rpath,{os.path.dirname(LIB)}", "-o", exe],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    return exe


def run(exe, grid, storage, tile, zseg, strips=0, fs=0, mutation=0):
    """(workgroups, violations), or None where the shape is refused."""
    args = [*grid, storage, tile, zseg, strips, fs, mutation]
    out = subprocess.run([exe, *map(str, args)], check=True, stdout=subprocess.PIPE, text=True).stdout
    f = out.strip().splitlines()[-1].split()
    if f[0] == "refused":
        return None
    assert f[0] == "blocks" and f[4] == "violations", out
    return int(f[1]), int(f[5])


GRIDS = [(29, 23, 26, 4), (17, 19, 18, 3), (40, 13, 15, 4), (11, 12, 13, 0), (64, 64, 9, 3), (65, 9, 11, 2),
         (127, 10, 12, 3), (131, 11, 9, 3), (257, 9, 9, 3), (300, 9, 10, 3), (9, 40, 31, 1), (254, 9, 9, 2), (13, 14, 15, 5)]


@pytest.mark.parametrize("grid", GRIDS)
def test_march_shapes(checker, grid):
    ran = 0
    for storage in (0, 2):
        for tile, zseg, strips in ((192, 1, 0), (256, 3, 2), (384, 64, 0), (512, 2, 3), (1024, 5, 0)):
            for fs in (0, 1):
                r = run(checker, grid, storage, tile, zseg, strips, fs)
                if r is None:  # too many workgroups, or too many threads for FP64
                    continue
                ran += 1
                assert r[0] > 0 and r[1] == 0, (storage, tile, zseg, strips, fs, r)
    assert ran >= 6


@pytest.mark.parametrize("grid", [(101, 641, 40, 10), (401, 101, 41, 10), (480, 60, 30, 10), (1024, 31, 24, 10)])
def test_march_workload_rows(checker, grid):
    for tile in (512, 768, 1024):
        r = run(checker, grid, 0, tile, 16)
        assert r is not None and r[1] == 0, (tile, r)


def test_checker_catches_mistakes(checker):
    for mutation in (1, 2):
        assert run(checker, (29, 23, 26, 4), 0, 256, 4, mutation=mutation)[1] > 0


@pytest.mark.parametrize("dims,storage,sets", [
    ((33, 33, 33), 0, 2), ((101, 101, 101), 0, 2), ((160, 160, 160), 0, 1), ((256, 256, 256), 0, 2),
    ((65, 800, 640), 0, 1), ((80, 800, 640), 0, 2), ((120, 120, 120), 2, 1), ((192, 200, 188), 2, 2),
    ((101, 101, 101), 1, 1), ((700, 700, 700), 0, 1)])
def test_schedule_by_rule(dims, storage, sets):
    """Which new shots take the whole-grid step: small grids, and those beyond the last-level
    cache with enough of a wave's lanes on columns; not FP16, nor sets of many gigabytes."""
    from helpers import small_cfg
    cfg = small_cfg(nx=dims[0], ny=dims[1], nz=dims[2], nstep=10, npml=10, storage=storage)
    one, two = cfg.replace(block=128, zseg=2).plan()["device_bytes"], cfg.plan()["device_bytes"]
    cells = dims[0] * dims[1] * dims[2]
    assert two == one if sets == 1 else two >= one + 9 * cells * (8 if storage == 2 else 4)
