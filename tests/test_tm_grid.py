"""The grid of the tiled z-march covers every shape that the operator entries
take, without a GPU: tests/cpp/tm_grid_check.cpp compiled for the host alone.

A plane of more than 65536 tiles of 64 x 8 cells can never meet the bound on
reduction partials by longer chunks; the search for one must end all the same
(it used to count on until the chunk overflowed)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SHAPES = [(48, 1, 1), (64, 8, 16), (65, 9, 17), (256, 256, 256), (4096, 4096, 1), (8192, 8192, 1),
          (8192, 8192, 16), (65535, 513, 3), (65535, 32767, 1), (48, 65535, 600)]


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path_factory.mktemp("tm") / "tm_grid_check")
    subprocess.run([HIPCC, "--offload-host-only", "-x", "hip", "-O1", "-std=c++17", "-w", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "tm_grid_check.cpp")], check=True)
    p = subprocess.run([exe], input="".join("%d %d %d\n" % s for s in SHAPES), text=True,
                       capture_output=True, timeout=20, check=True)
    return [tuple(int(v) for v in line.split()) for line in p.stdout.splitlines()]


@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_tm_grid_covers_the_shape(grids, i):
    nx, ny, nz = SHAPES[i]
    gx, gy, gz, zc = grids[i]
    assert (gx, gy) == (-(-nx // 64), -(-ny // 8))
    assert 1 <= zc <= nz and gz == -(-nz // zc)
    assert gx * gy * gz <= 65536 or zc == nz
