"""flowhip_run and flowhip_run_f32 keep several steps in flight; the driver
loop of main.c:64-115 looks at dt after every step. Both stop after the same
step and leave the same state: a run with sim_end inside it, more steps than
may be in flight at once, and a run continued from another one, against the
same steps taken one call at a time."""
import numpy as np
import pytest

import flow_amd
from flow_amd import problems

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "e", "u", "v", "mom_x", "mom_y")


def _state(n, fp32, sim_end=1.0e30):
    m = flow_amd.Mesh(n, n, dt=2.0e-4, sim_end=sim_end)
    st = flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m)
    rho, e = problems.sod_x(n)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    return m, st


def _one_by_one(n, fp32, steps, sim_end=1.0e30):
    m, st = _state(n, fp32)
    pairs, totals, elapsed, k = [], [], 0.0, 0
    while k < steps:
        done, dt, mass, energy, _ = st.run(1, tt0=k, pre_timestep=(k == 0))
        assert done == 1
        if k == 0:
            pairs.append(dt[0])
        pairs.append(dt[1])
        totals.append((mass[0], energy[0]))
        elapsed += dt[1][0]
        k += 1
        if elapsed >= sim_end:
            break
    fields = {f: st.download(f) for f in FIELDS}
    st.close()
    m.close()
    return k, np.array(pairs), np.array(totals), fields


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n,steps,stop", [(33, 20, 7), (48, 20, 1), (40, 150, 131),
                                          (64, 130, None)])
def test_run_equals_single_steps(n, steps, stop, fp32):
    print(f"case run-ahead n={n} steps={steps} stop={stop} fp32={fp32}", flush=True)
    sim_end = 1.0e30
    if stop:
        _, pairs, _, _ = _one_by_one(n, fp32, stop)
        # between the times after stop - 1 and stop steps
        sim_end = float(pairs[1:stop, 0].sum() + 0.5 * pairs[stop, 0])
    want = _one_by_one(n, fp32, steps, sim_end)
    m, st = _state(n, fp32, sim_end)
    done, dt, mass, energy, _ = st.run(steps)
    assert done == want[0] == (stop or steps)
    assert np.array_equal(dt, want[1])
    assert np.array_equal(np.stack([mass, energy], 1), want[2])
    for f in FIELDS:
        assert np.array_equal(st.download(f), want[3][f]), f
    st.close()
    m.close()
