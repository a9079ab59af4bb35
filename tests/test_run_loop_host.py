"""The order in which flowhip_run's loop puts work on the stream and waits for
it, on the host alone (tests/hostcheck/run_loop_host.c): whatever it puts there
it waits for before it returns, the upload of the dt pair among it, whose pinned
buffer and whose values are the caller's next call's."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "hostcheck", "run_loop_host.c")


@pytest.fixture(scope="module")
def run_log(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("run_loop") / "run_loop_host.so")
    rocm = os.environ.get("ROCM", "/opt/rocm")
    # what the loop itself does not call stays unresolved
    subprocess.run(["gcc", "-O1", "-std=gnu99", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    f"-I{rocm}/include", "-Wl,-z,lazy,-Bsymbolic", SRC, "-o", so],
                   check=True, capture_output=True, timeout=300)
    fn = ctypes.CDLL(so, mode=os.RTLD_LAZY | os.RTLD_LOCAL).run_log
    fn.restype = ctypes.c_char_p
    return lambda *a: fn(*a).decode()


def test_nothing_to_do_does_nothing(run_log):
    assert run_log(0, 0, 0) == ""


@pytest.mark.parametrize("niters,tt0,pre,want", [
    (0, 0, 1, "PBWT"), (1, 0, 0, "PSWT"), (3, 0, 1, "PBWTSSSWTTT"), (3, -2, 1, "PBWTSSSWTTT"),
    (3, -9, 0, "PSSSWTTT"), (70, 0, 0, "P" + "S" * 64 + "W" + "T" * 64 + "SSSSSSWTTTTTT")])
def test_every_launch_is_waited_for(run_log, niters, tt0, pre, want):
    assert run_log(niters, tt0, pre) == want
