"""The march launchers refuse a mesh without interior cells (hipErrorInvalidValue
before anything is launched), and the division-free strip quotient refuses no
strips: both once divided by the number of strips, zero. Runs without a GPU (hidden
where there is one), each case in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INVALID_VALUE = 1


def _python(code):
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                          timeout=300, env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"))


CODE = """
import sys
sys.path.insert(0, %r)
from tests import kernel_abi as abi
L = abi.lib()
nx, ny, rows, pairs = %d, %d, %d, %d
out = []
for fp32 in (False, True):
    m = abi.mesh(fp32, nx, ny, pairs)
    for tt in (0, 1):
        out += abi.march_calls(L, m, fp32, tt, rows)
print(*out)
"""


@pytest.mark.parametrize("rows", [0, 16])
@pytest.mark.parametrize("nx,ny,pairs", [(4, 40, 1), (40, 4, 1), (4, 4, 1), (3, 40, 1), (0, 0, 1),
                                         (-8, 40, 1), (-90, -90, 1), (4, 40, 2)])
def test_march_launchers_refuse_an_empty_interior(nx, ny, pairs, rows):
    r = _python(CODE % (ROOT, nx, ny, rows, pairs))
    assert r.returncode == 0, (r.returncode, r.stderr)
    got = [int(v) for v in r.stdout.split()]
    assert got and set(got) == {INVALID_VALUE}


@pytest.mark.parametrize("n", [0, -1])
def test_strip_inverse_of_no_strips(n):
    code = ("import ctypes, sys; sys.path.insert(0, %r); from tests import kernel_abi as abi;"
            "f = abi.lib().fk_strip_inverse; f.restype = ctypes.c_ulonglong; print(f(%d))"
            % (ROOT, n))
    r = _python(code)
    assert r.returncode == 0 and r.stdout.split() == ["0"], (r.returncode, r.stderr)
