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


# (nx, ny) of indexable fields whose lists pass the strip quotient's bounds
@pytest.mark.parametrize("nx,ny,rows", [(300_000_006, 6, 0), (300_000_006, 6, 4),
                                        (5, 350_000_000, 4)])
def test_march_launchers_refuse_lists_past_the_strip_quotient(nx, ny, rows):
    r = _python(CODE % (ROOT, nx, ny, rows, 0))
    assert r.returncode == 0, (r.returncode, r.stderr)
    got = [int(v) for v in r.stdout.split()]
    assert got and set(got) == {INVALID_VALUE}


def test_strip_quotient_within_its_bounds():
    """item / n as the kernels form it, in 64 bits, at both bounds."""
    code = ("import ctypes, sys; sys.path.insert(0, %r); from tests import kernel_abi as abi;"
            "f = abi.lib().fk_strip_inverse; f.restype = ctypes.c_ulonglong;"
            "print(*[f(n) for n in %r])")
    counts = [1, 2, 3, 7, 58, 799, 800, 1021, 65535, 300001]
    r = _python(code % (ROOT, counts))
    assert r.returncode == 0, r.stderr
    for n, inv in zip(counts, map(int, r.stdout.split())):
        last = min(2 ** 24 * n, (2 ** 40 - 1) // n, 2 ** 31 - 1) - 1
        for item in {0, 1, n - 1, n, n + 1, last // n * n - 1, last // n * n, last}:
            if 0 <= item <= last:
                assert ((item * inv) % 2 ** 64) >> 40 == item // n, (n, item)
