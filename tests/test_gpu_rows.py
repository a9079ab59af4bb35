"""The row-parallel kernels of small meshes against the marches on the same
inputs (a given chunk height asks for the march): every array and the dt
sequence bit for bit, over strips and row blocks with every remainder, from the
smallest mesh to the sizes where the forms meet, on uniform meshes and on meshes
whose spacings differ (powers of two or not), FP64 and FP32 state.

The totals are sums of the same cells grouped by other items: a lane's sum is
rounded once a group (FP64 state, compensated sums; 2^-53 each way, and the
total's own rounding), or within 240 roundings (FP32 state, plain FP64 sums).
"""
import ctypes

import numpy as np
import pytest

import flow_amd
from flow_amd import native, problems

pytestmark = pytest.mark.gpu

SIZES = [(2, 2), (2, 3), (57, 12), (58, 3), (59, 61), (60, 14), (61, 16), (64, 64), (117, 45),
         (181, 128), (640, 9), (3, 700), (500, 430), (700, 690)]


def _spacings(kind, mesh):
    """Overwrites the mesh's device spacings, cell and edge, along both axes."""
    if kind == "uniform":
        return
    rng = np.random.default_rng(7)
    for name, n in (("edgedx", mesh.nx), ("edgedy", mesh.ny), ("celldx", mesh.nx),
                    ("celldy", mesh.ny)):
        if kind == "pow2":
            d = 2.0 ** -rng.integers(6, 8, n + 1)
        else:
            d = 0.01 * rng.uniform(0.7, 1.4, n + 1)
        d = np.ascontiguousarray(d, dtype=np.float64)
        ptr = getattr(mesh.s, name)
        native.lib().flowhip_copy(ctypes.cast(ptr, ctypes.c_void_p),
                                  d.ctypes.data_as(ctypes.c_void_p), n + 1, native.SEND)


def _run(nx, ny, kind, fp32, march_rows, steps=4):
    m = flow_amd.Mesh(nx, ny, dt=1.0e-5)
    m.set_schedule(flow_amd.MARCH)
    _spacings(kind, m)
    if march_rows:
        m.set_march_rows(march_rows)
    st = flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m)
    rho, e = problems.boxes(nx, ny, [(1.0, 0.25, 0.0, 0.0, 1.0, 1.0),
                                     (1.0, 25.0, 0.3, 0.4, 0.2, 0.25),
                                     (0.5, 5.0, 0.6, 0.0, 0.4, 0.3)])
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    done, dts, mass, energy, _ = st.run(steps)
    out = dict(arrays=st.download_all(), dt=dts, mass=mass, energy=energy)
    assert done == steps
    st.close()
    m.close()
    return out


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("kind", ["uniform", "pow2", "any"])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_rows_equal_march(nx, ny, kind, fp32):
    print(f"case {nx}x{ny} {kind} fp32={fp32}", flush=True)
    a = _run(nx, ny, kind, fp32, 0)
    b = _run(nx, ny, kind, fp32, 16)
    for k in b["arrays"]:
        ndiff = int(np.count_nonzero(a["arrays"][k].view(np.uint8) !=
                                     b["arrays"][k].view(np.uint8)))
        assert ndiff == 0, (k, ndiff)
    np.testing.assert_array_equal(a["dt"], b["dt"])
    rtol = (2 * 240 + 2 if fp32 else 6) * 2.0 ** -53
    np.testing.assert_allclose(a["mass"], b["mass"], rtol=rtol, atol=0)
    np.testing.assert_allclose(a["energy"], b["energy"], rtol=rtol, atol=0)
