"""Spacings written into a mesh's own arrays after its first step count from the
next call on once flowhip_geometry_changed has been called: the run goes on as on
a mesh that held them from the start."""
import ctypes

import numpy as np
import pytest

import flow_amd
from flow_amd import native, problems

pytestmark = pytest.mark.gpu

NX, NY = 70, 41
EDITS = {
    "cells": {"celldx": 0.02, "celldy": 0.031},
    "all": {"edgedx": 0.02, "edgedy": 0.031, "celldx": 0.02, "celldy": 0.031},
    "pow2": {"edgedx": 1 / 64, "edgedy": 1 / 32, "celldx": 1 / 64, "celldy": 1 / 32},
    "varied": {"celldy": None, "edgedy": None},
}


def _edit(m, kind):
    rng = np.random.default_rng(3)
    for name, value in EDITS[kind].items():
        n = (m.nx if name.endswith("x") else m.ny) + 1
        d = np.full(n, value) if value else 0.02 * rng.uniform(0.8, 1.3, n)
        native.lib().flowhip_copy(ctypes.cast(getattr(m.s, name), ctypes.c_void_p),
                                  d.ctypes.data_as(ctypes.c_void_p), n, native.SEND)


def _mesh(fp32):
    m = flow_amd.Mesh(NX, NY, dt=1.0e-4)
    return m, (flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m))


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("rows", [0, 16])
@pytest.mark.parametrize("kind", list(EDITS))
def test_edited_spacings_count(kind, rows, fp32):
    print(f"case geometry changed {kind} rows={rows} fp32={fp32}", flush=True)
    rho, e = problems.boxes(NX, NY, [(1.0, 0.25, 0.0, 0.0, 1.0, 1.0),
                                     (1.0, 25.0, 0.3, 0.4, 0.2, 0.25)])
    m, st = _mesh(fp32)
    m.set_march_rows(rows)
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    st.run(3)
    fresh, fs = _mesh(fp32)
    fresh.set_march_rows(rows)
    _edit(fresh, kind)
    for k, a in st.download_all().items():
        fs.upload(k, a)
    fresh.set_dt(m.dt, m.dt_h)
    _edit(m, kind)
    m.geometry_changed()
    for pre in (True, False):
        a = st.run(3, tt0=3, pre_timestep=pre)
        b = fs.run(3, tt0=3, pre_timestep=pre)
        for x, y in zip(a[:4], b[:4]):
            np.testing.assert_array_equal(x, y)
    for k, a in st.download_all().items():
        np.testing.assert_array_equal(a, fs.download(k), err_msg=k)
    for s, x in ((st, m), (fs, fresh)):
        s.close()
        x.close()
