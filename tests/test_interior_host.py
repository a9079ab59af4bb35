"""The cells that set_timestep and print_conservation visit: the interior of the
nx x ny local array they are given, in row-major order, and none where the pad
leaves no interior (the caller gives the sizes). Compiled for the host."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "hostcheck", "interior_host.cpp")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

EMPTY = [(3, 100), (100, 3), (3, 3), (4, 9), (9, 4), (0, 0), (0, 50), (50, 0), (1, 2), (-5, 7),
         (7, -5), (-9, -9)]
SIZES = [(5, 5), (6, 5), (5, 9), (40, 20), (61, 66)]
# the largest mesh: an index and the stride of a grid past it fit 32 bits
LARGEST = 46335


@pytest.fixture(scope="module")
def interior(tmp_path_factory):
    if not shutil.which(HIPCC) and not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    exe = str(tmp_path_factory.mktemp("interior") / "interior_host")
    subprocess.run([HIPCC, "-O2", "-std=c++17", SRC, "-o", exe], check=True,
                   capture_output=True, timeout=600)

    def run(nx, ny):
        out = subprocess.run([exe], input=f"{nx} {ny} 2\n", capture_output=True, text=True,
                             check=True, timeout=60).stdout.split()
        return int(out[0]), [tuple(int(v) for v in c.split(",")) for c in out[1:]]
    return run


@pytest.mark.parametrize("nx,ny", EMPTY)
def test_no_interior_no_cells(interior, nx, ny):
    assert interior(nx, ny) == (0, [])


@pytest.mark.parametrize("nx,ny", SIZES)
def test_every_interior_cell_once(interior, nx, ny):
    want = [(i, j) for i in range(2, ny - 2) for j in range(2, nx - 2)]
    assert interior(nx, ny) == (len(want), want)


def test_largest_mesh(interior):
    n, _ = interior(LARGEST + 4, LARGEST + 4)
    assert n == LARGEST ** 2 < 2 ** 31
