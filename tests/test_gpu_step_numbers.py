"""flowhip_run, flowhip_run_f32 and the ensemble take any step number, as
solve_hydro_2d does: tt counts (below zero too) only by its parity and by
tt == 0's first-step update of dt_h (omp3/flow.c:103-105, 307, 565)."""
import numpy as np
import pytest

import flow_amd
from flow_amd import problems

pytestmark = pytest.mark.gpu

N = 48
FIELDS = ("rho", "e", "u", "v", "mom_x", "mom_y")


def _state(fp32):
    m = flow_amd.Mesh(N, N, dt=2.0e-4)
    st = flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m)
    rho, e = problems.sod_x(N)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    return m, st


def _result(m, st, out):
    res = (out[0], out[1], np.stack(out[2:4], 1), {f: st.download(f) for f in FIELDS})
    st.close()
    m.close()
    return res


def _same(a, b):
    assert a[0] == b[0]
    np.testing.assert_array_equal(a[1], b[1])
    np.testing.assert_array_equal(a[2], b[2])
    for f in FIELDS:
        np.testing.assert_array_equal(a[3][f], b[3][f], err_msg=f)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("tt0", [-3, -70])
def test_run_below_step_zero(tt0, fp32):
    """Steps below zero are steps of their parity."""
    print(f"case run tt0={tt0} fp32={fp32}", flush=True)
    steps = min(-tt0, 68)
    got, want = _state(fp32), _state(fp32)
    a = _result(*got, got[1].run(steps, tt0=tt0))
    b = _result(*want, want[1].run(steps, tt0=100 + tt0 % 2))
    _same(a, b)


def test_run_through_step_zero():
    """The same calls as solve_hydro_2d, one a step."""
    print("case run -3 .. 3 against solve_hydro_2d", flush=True)
    m, st = _state(False)
    _, dts, _, _, _ = st.run(7, tt0=-3)
    fields = {f: st.download(f) for f in FIELDS}
    st.close()
    m.close()
    m, st = _state(False)
    st.set_timestep(0)
    want = [(m.dt, m.dt_h)]
    for tt in range(-3, 4):
        st.solve(tt)
        want.append((m.dt, m.dt_h))
    np.testing.assert_array_equal(dts, want)
    for f in FIELDS:
        np.testing.assert_array_equal(fields[f], st.download(f), err_msg=f)
    st.close()
    m.close()


@pytest.mark.parametrize("tt0", [-6, -5, -4, -3, -2, -1, 0])
def test_ensemble_replays_around_step_zero(tt0):
    """Replayed steps equal direct ones, where the first run passes step zero
    and the second replays what the first captured."""
    print(f"case ensemble tt0={tt0}", flush=True)
    sizes = [33, 64]
    out = []
    for graphs in (False, True):
        ens = flow_amd.Ensemble(sizes, dt=2.0e-4)
        for k, n in enumerate(sizes):
            ens.set_state(k, *problems.sod_x(n))
        ens.set_graphs(graphs)
        runs = [ens.run(12, tt0=tt0)[:3],
                ens.run(13, tt0=tt0 + 12, pre_timestep=False)[:3]]
        out.append((runs, [ens.get(k, f) for k in range(2) for f in FIELDS]))
        ens.close()
    for a, b in zip(out[0][0], out[1][0]):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)
    for x, y in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(x, y)
