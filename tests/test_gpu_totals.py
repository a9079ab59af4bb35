"""print_conservation and flowhip_run give the totals of the state as it is,
also where the step before them ran under another schedule than the one before
that: the march and fused steps leave totals for the next print_conservation,
the stagewise step leaves none.

The totals are compensated FP64 sums of rho and of the rounded products rho e:
one rounding of the sum (2^-53) and second-order terms, against the exact sums
of the same values."""
import ctypes
import math

import numpy as np
import pytest

import flow_amd
from flow_amd import native, problems

pytestmark = pytest.mark.gpu

N = 48
RTOL = 4 * 2.0 ** -53


def _state():
    m = flow_amd.Mesh(N, N, dt=2.0e-4)
    st = flow_amd.DeviceState(m)
    rho, e = problems.sod_x(N)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    st.set_timestep(0)
    return m, st


def _close(m, st):
    st.close()
    m.close()


def _last_sums(m):
    fn = native.lib().flowhip_last_sums
    fn.argtypes = [ctypes.c_void_p] + [ctypes.POINTER(ctypes.c_double)] * 2
    mass, energy = ctypes.c_double(), ctypes.c_double()
    fn(m.ptr, ctypes.byref(mass), ctypes.byref(energy))
    return mass.value, energy.value


def _print_conservation(m, st):
    native.lib().print_conservation(m.nx, m.ny, ctypes.c_void_p(st.ptrs["rho"]),
                                    ctypes.c_void_p(st.ptrs["e"]), None, m.ptr)
    return _last_sums(m)


def _exact(m, st):
    L = m.nx
    inner = (slice(2, -2), slice(2, -2))
    rho = st.download("rho")[: L * L].reshape(L, L)[inner]
    e = st.download("e")[: L * L].reshape(L, L)[inner]
    return math.fsum(rho.ravel()), math.fsum((rho * e).ravel())


@pytest.mark.parametrize("first", [flow_amd.MARCH, flow_amd.FUSED])
def test_totals_follow_a_change_of_schedule(first):
    print(f"case totals schedule {first} then stagewise", flush=True)
    m, st = _state()
    m.set_schedule(first)
    st.solve(0)
    m.set_schedule(flow_amd.STAGEWISE)
    st.solve(1)
    got = _print_conservation(m, st)
    np.testing.assert_allclose(got, _exact(m, st), rtol=RTOL, atol=0)
    m.set_schedule(first)
    st.solve(2)
    got = _print_conservation(m, st)
    np.testing.assert_allclose(got, _exact(m, st), rtol=RTOL, atol=0)
    _close(m, st)


def test_printed_run_after_another_schedule(capfd):
    print("case totals march then a printed stagewise run", flush=True)
    m, st = _state()
    st.solve(0)
    m.set_schedule(flow_amd.STAGEWISE)
    m.s.verbose = 1
    _, _, mass, energy, _ = st.run(1, tt0=1, pre_timestep=False)
    m.s.verbose = 0
    np.testing.assert_allclose((mass[0], energy[0]), _exact(m, st), rtol=RTOL, atol=0)
    _close(m, st)


def test_last_totals_stay_until_the_next_ones():
    """A step that leaves no totals leaves the last ones as they were."""
    print("case last totals after a run, then a stagewise step", flush=True)
    m, st = _state()
    _, _, mass, energy, _ = st.run(5, tt0=0, pre_timestep=False)
    assert _last_sums(m) == (mass[-1], energy[-1])
    m.set_schedule(flow_amd.STAGEWISE)
    st.solve(5)
    assert _last_sums(m) == (mass[-1], energy[-1])
    _close(m, st)


@pytest.mark.parametrize("rule", [flow_amd.CFL_DEFINED, flow_amd.CFL_OMP3_SERIAL])
@pytest.mark.parametrize("nx,ny", [(3, 40), (40, 3), (4, 40), (2, 2)])
def test_no_interior(nx, ny, rule):
    """Sizes without interior cells: totals of nothing, and the dt pair that
    max_dt and dt_h give (C_T 0.3, C_M 5: omp3/flow.c:103-105)."""
    print(f"case no interior {nx}x{ny} rule={rule}", flush=True)
    m, st = _state()
    m.set_cfl_rule(rule)
    m.s.max_dt = 1.0e-3
    m.set_dt(3.0e-4, 4.0e-4)
    arg = {k: ctypes.c_void_p(st.ptrs[k]) for k in ("Qxx", "Qyy", "rho", "e")}
    native.lib().set_timestep(nx, ny, arg["Qxx"], arg["Qyy"], arg["rho"], arg["e"], m.ptr, None,
                              0, ctypes.cast(m.s.celldx, ctypes.c_void_p),
                              ctypes.cast(m.s.celldy, ctypes.c_void_p))
    least = min(1.0e-3, (1.5 / 0.3) * 4.0e-4)
    assert (m.dt, m.dt_h) == (0.5 * (0.3 * least + 4.0e-4), 0.3 * least)
    native.lib().print_conservation(nx, ny, arg["rho"], arg["e"], None, m.ptr)
    assert _last_sums(m) == (0.0, 0.0)
    _close(m, st)
