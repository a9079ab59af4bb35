"""A replayed step uses the spacings its mesh has now, as a direct step does: a
mesh pointed at other spacing arrays and back at the first ones, which hold other
values by then."""
import ctypes

import numpy as np
import pytest

import flow_amd
from flow_amd import native, problems

pytestmark = pytest.mark.gpu

N = 48
NAMES = ("edgedx", "edgedy", "celldx", "celldy")
FIELDS = ("rho", "e", "u", "v", "mom_x", "mom_y")


def _fill(ptr, value):
    d = np.full(N + 5, value)
    native.lib().flowhip_copy(ctypes.c_void_p(ptr), d.ctypes.data_as(ctypes.c_void_p), N + 5,
                              native.SEND)


def _point(m, ptrs):
    for k in NAMES:
        setattr(m.s, k, ctypes.cast(ptrs[k], ctypes.POINTER(ctypes.c_double)))


def _steps(graphs, back_to):
    m = flow_amd.Mesh(N, N, dt=1.0e-4)
    m.set_graphs(graphs)
    st = flow_amd.DeviceState(m)
    rho, e = problems.sod_x(N)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    own = {k: ctypes.cast(getattr(m.s, k), ctypes.c_void_p).value for k in NAMES}
    other = {}
    for k in NAMES:
        p = ctypes.c_void_p()
        native.lib().allocate_data(ctypes.byref(p), N + 5)
        other[k] = p.value
        _fill(p.value, 0.03)
    st.set_timestep(0)
    for tt in range(1, 5):
        st.solve(tt)
    _point(m, other)
    st.solve(5)
    for k in NAMES:
        _fill(own[k], back_to)
    _point(m, own)
    pairs = []
    for tt in range(6, 10):
        st.solve(tt)
        pairs.append((m.dt, m.dt_h))
    out = (pairs, {f: st.download(f) for f in FIELDS})
    for p in other.values():
        native.lib().deallocate_data(ctypes.c_void_p(p))
    st.close()
    m.close()
    return out


# the second keeps every geometry flag of the first arrays' old values, 1 / 48
@pytest.mark.parametrize("back_to", [1.0 / 64, 0.05])
def test_replayed_steps_follow_the_spacings(back_to):
    print(f"case graph geometry back_to={back_to}", flush=True)
    a, b = _steps(True, back_to), _steps(False, back_to)
    assert a[0] == b[0]
    for f in FIELDS:
        assert np.array_equal(a[1][f], b[1][f]), f
