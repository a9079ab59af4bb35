"""The march kernels themselves (small meshes take their row-parallel form
unless a chunk height is given) in every geometry form, and at the chunk heights
that they choose just above the sizes where they take over.

Every array and the dt sequence bit for bit: the forms among each other at given
heights; the chosen heights against given ones and, in FP64, the oracle. The
totals are sums of the same cells in other groups: rounded once a group (2^-53
each way, and the total's own rounding), or within 240 roundings (FP32 state)."""
import numpy as np
import pytest

import flow_amd
from flow_amd import problems
from tests import harness

pytestmark = pytest.mark.gpu

FORMS = {"uniform": {}, "loaded": {"FLOWHIP_UNIFORM": "0"}, "ieee": {"FLOWHIP_POW2": "0"},
         "loaded ieee": {"FLOWHIP_UNIFORM": "0", "FLOWHIP_POW2": "0"}}
BOXES = [(1.0, 0.25, 0.0, 0.0, 1.0, 1.0), (1.0, 25.0, 0.3, 0.4, 0.2, 0.25),
         (0.5, 5.0, 0.6, 0.0, 0.4, 0.3)]


def _run(monkeypatch, env, nx, ny, rows, fp32, steps):
    for k in ("FLOWHIP_UNIFORM", "FLOWHIP_POW2"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    m = flow_amd.Mesh(nx, ny, dt=1.0e-5)
    m.set_schedule(flow_amd.MARCH)
    m.set_march_rows(rows)
    st = flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m)
    rho, e = problems.boxes(nx, ny, BOXES)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    done, dts, mass, energy, _ = st.run(steps)
    assert done == steps
    out = dict(arrays=st.download_all(), dt=dts, mass=mass, energy=energy)
    st.close()
    m.close()
    return out


def _same(a, b, fp32):
    for k in b["arrays"]:
        ndiff = int(np.count_nonzero(a["arrays"][k].view(np.uint8) !=
                                     b["arrays"][k].view(np.uint8)))
        assert ndiff == 0, (k, ndiff)
    np.testing.assert_array_equal(a["dt"], b["dt"])
    rtol = (2 * 240 + 2 if fp32 else 6) * 2.0 ** -53
    np.testing.assert_allclose(a["mass"], b["mass"], rtol=rtol, atol=0)
    np.testing.assert_allclose(a["energy"], b["energy"], rtol=rtol, atol=0)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("rows", [4, 20])
@pytest.mark.parametrize("nx,ny", [(256, 256), (128, 256), (192, 96), (190, 131)])
def test_march_geometry_forms_agree(monkeypatch, nx, ny, rows, fp32):
    print(f"case march forms {nx}x{ny} rows={rows} fp32={fp32}", flush=True)
    base = _run(monkeypatch, {}, nx, ny, 0, fp32, 4)
    for name, env in FORMS.items():
        print(f"  {name}", flush=True)
        _same(_run(monkeypatch, env, nx, ny, rows, fp32, 4), base, fp32)


# none a power of two: with 256 CUs the FP64 and FP32 marches take over, one
# kernel after the other, between the first and the last
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("nx,ny", [(690, 710), (730, 730), (790, 850), (850, 850), (951, 949)])
def test_chosen_march_heights(monkeypatch, nx, ny, fp32):
    print(f"case march heights {nx}x{ny} fp32={fp32}", flush=True)
    steps = 4
    a = _run(monkeypatch, {}, nx, ny, 0, fp32, steps)
    _same(a, _run(monkeypatch, {}, nx, ny, 16, fp32, steps), fp32)
    if not fp32:
        ref = harness.oracle_run(None, (nx, ny), steps, dt=1.0e-5,
                                 init=problems.boxes(nx, ny, BOXES))
        for k, (rel, ndiff) in harness.compare_state(a["arrays"], ref["arrays"],
                                                     ref["L"]).items():
            assert ndiff == 0, (k, rel, ndiff)
        np.testing.assert_array_equal(a["dt"], ref["dt"])
