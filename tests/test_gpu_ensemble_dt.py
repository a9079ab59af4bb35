"""The dt pairs and totals of an ensemble, which its march kernels hand to each
other (one CFL word per instance, totals folded at the front of the momentum
march), against the same meshes alone: states at rest (every candidate equal),
undefined candidates, a binding max_dt, numbers of instances around the four
waves of a block, both momentum schedules, direct and replayed, several runs in
a row on one ensemble.

dt pairs and counts are the same bits; the totals are the same compensated
sums in other groups (rounded once a group, 2^-53 each, and once at the end)."""
import numpy as np
import pytest

import flow_amd
from flow_amd import problems

pytestmark = pytest.mark.gpu

SIZES = [33, 2, 64, 130, 17, 58, 59, 90, 121]
STEPS = 6


def _init(kind, k, n):
    if kind == "blast":
        return problems.ensemble_instance(n, "blast", 0.3 + 0.05 * k, 10.0 * (k + 1))
    rho, e = problems.boxes(n, n, [(1.0, 2.5, 0.0, 0.0, 1.0, 1.0)])
    if kind == "undefined":
        L = problems.local_size(n)
        rng = np.random.default_rng(k)
        i, j = rng.integers(2, 2 + n, 3), rng.integers(2, 2 + n, 3)
        e[i * L + j] = -1.0
    return rho, e


def _single(kind, k, n, fp32, max_dt):
    m = flow_amd.Mesh(n, n, dt=1.0e-4, max_dt=max_dt)
    m.set_schedule(flow_amd.MARCH)
    st = flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m)
    rho, e = _init(kind, k, n)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    out = []
    for r in range(2):
        _, dts, mass, energy, _ = st.run(STEPS, tt0=r * STEPS, pre_timestep=r == 0)
        out.append((dts, mass, energy, st.undefined))
    st.close()
    m.close()
    return out


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("count,fused,graphs", [(1, True, False), (5, False, True),
                                                (9, True, True)])
@pytest.mark.parametrize("kind,max_dt", [("rest", 1.0e30), ("undefined", 1.0e30),
                                         ("blast", 1.0e30), ("blast", 2.0e-5)])
def test_ensemble_steps_equal_single_meshes(kind, max_dt, count, fused, graphs, fp32):
    print(f"case {kind} max_dt={max_dt} count={count} fused={fused} graphs={graphs} "
          f"fp32={fp32}", flush=True)
    sizes = SIZES[:count] if kind != "undefined" else [n for n in SIZES if n > 8][:count]
    ens = flow_amd.Ensemble(sizes, dt=1.0e-4, max_dt=max_dt, fp32=fp32)
    for k, n in enumerate(sizes):
        ens.set_state(k, *_init(kind, k, n))
    ens.set_schedule(8, 1, fused)
    ens.set_graphs(graphs)
    got = []
    for r in range(2):
        dts, mass, energy, _ = ens.run(STEPS, tt0=r * STEPS, pre_timestep=r == 0)
        got.append((dts, mass, energy, ens.undefined))
    ens.close()
    for k, n in enumerate(sizes):
        for g, w in zip(got, _single(kind, k, n, fp32, max_dt)):
            np.testing.assert_array_equal(g[0][k], w[0])
            np.testing.assert_array_equal(g[3][k], w[3][-STEPS:])
            rtol = (2 * 240 + 2 if fp32 else 6) * 2.0 ** -53
            np.testing.assert_allclose(g[1][k], w[1], rtol=rtol, atol=0)
            np.testing.assert_allclose(g[2][k], w[2], rtol=rtol, atol=0)
