"""A march step through the kernel launchers with the momentum directions apart
(fk_march_momentum_x, then _y) against flowhip_run, whose steps take both in one
march: every array the step leaves, the dt pair and the totals bit for bit, FP64
and FP32 state, both sweep orders and the first step's dt update, with and
without power-of-two spacings."""
import ctypes

import numpy as np
import pytest

import flow_amd
from flow_amd import native, problems
from tests import kernel_abi as abi

pytestmark = pytest.mark.gpu

ROWS = 16  # the same chunks on both sides, so the same totals
STEPS = 5
FIELDS = ("rho", "e", "u", "v", "mom_x", "mom_y", "F_x", "F_y", "rho_old")


def _state(nx, ny, fp32):
    m = flow_amd.Mesh(nx, ny, dt=1.0e-4)
    m.set_march_rows(ROWS)
    st = flow_amd.DeviceState32(m) if fp32 else flow_amd.DeviceState(m)
    rho, e = problems.boxes(nx, ny, [(1.0, 0.25, 0.0, 0.0, 1.0, 1.0),
                                     (1.0, 25.0, 0.3, 0.4, 0.2, 0.25)])
    st.upload("rho", rho)
    st.upload("e", e)
    st.reflect_initial()
    st.run(0)  # the pre-loop time step
    return m, st


class _Buffers:
    """Zeroed device doubles."""

    def __init__(self):
        self.all = []

    def new(self, n):
        p = ctypes.c_void_p()
        native.lib().allocate_data(ctypes.byref(p), n)
        self.all.append(p)
        return p.value

    def free(self):
        for p in self.all:
            native.lib().deallocate_data(p)


def _read(ptr, n):
    out = np.empty(n)
    native.lib().flowhip_copy(ctypes.c_void_p(ptr), out.ctypes.data_as(ctypes.c_void_p), n,
                              native.RECV)
    return out


def _geometry(L, b, m, fp32, pow2):
    """The mesh's spacings and their reciprocals, as the launchers take them."""
    ptrs = [ctypes.cast(getattr(m.s, k), ctypes.c_void_p).value
            for k in ("edgedx", "edgedy", "celldx", "celldy")]
    lens = [m.nx + 1, m.ny + 1] * 3
    for k in range(2):
        ptrs.append(b.new(lens[k]))
        assert L.fk_reciprocal(lens[k], ctypes.c_void_p(ptrs[4 + k]), ctypes.c_void_p(ptrs[k]),
                               None) == 0
    if fp32:
        wide, ptrs = ptrs, [b.new(n) for n in lens]
        for n, d, s in zip(lens, ptrs, wide):
            assert L.fk_narrow(ctypes.c_long(n), ctypes.c_void_p(d), ctypes.c_void_p(s),
                               None) == 0
    return abi.FkMesh(m.nx, m.ny, 2, *ptrs, pow2, 0, abi.FkUniform(), 0)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("nx,ny,pow2", [(61, 38, 0), (130, 77, 0), (128, 64, 1)])
def test_split_momentum_equals_one_march(nx, ny, pow2, fp32):
    print(f"case split momentum {nx}x{ny} pow2={pow2} fp32={fp32}", flush=True)
    L, b = abi.lib(), _Buffers()
    ma, sa = _state(nx, ny, fp32)
    _, dts, mass, energy, _ = sa.run(STEPS, pre_timestep=False)
    m, st = _state(nx, ny, fp32)
    geo = _geometry(L, b, m, fp32, pow2)
    r = abi.FkReduce(partials=b.new(L.fk_reduce_blocks()), dtp=b.new(4), sums=b.new(4),
                     status=b.new(4), queue=b.new(abi.QUEUE_WORDS // 2))
    pair = np.array([m.dt, m.dt_h])
    native.lib().flowhip_copy(ctypes.c_void_p(r.dtp), pair.ctypes.data_as(ctypes.c_void_p), 2,
                              native.SEND)
    native.sync()
    p, f = st.ptrs, "_f32" if fp32 else ""
    lag, parts = ctypes.c_int(), ctypes.c_int()
    for tt in range(STEPS):
        err = [
            getattr(L, "fk_march_lagrangian" + f)(
                geo, *[p[k] for k in ("rho", "e", "mom_x", "mom_y", "Qxx", "Qyy", "uF_x", "uF_y",
                                      "P", "rho_old")], r, 1.0e30, ctypes.byref(lag), ROWS, None),
            getattr(L, "fk_march_mass_energy" + f)(
                geo, tt, *[p[k] for k in ("uF_x", "uF_y", "rho_old", "P", "rho", "e", "F_x",
                                          "F_y")], r, 1.0e30, int(tt == 0), lag,
                ctypes.byref(parts), ROWS, None),
            getattr(L, "fk_march_momentum_x" + f)(
                geo, tt, *[p[k] for k in ("uF_x", "uF_y", "F_x", "F_y", "rho", "Qxx", "mom_x",
                                          "u")], r, ROWS, None),
            getattr(L, "fk_march_momentum_y" + f)(
                geo, tt, *[p[k] for k in ("u", "uF_y", "F_x", "F_y", "rho", "Qyy", "mom_y",
                                          "v")], r, parts, ROWS, None)]
        assert err == [0] * 4
        native.sync()
        assert np.array_equal(_read(r.dtp, 2), dts[tt + 1]), tt
        assert np.array_equal(_read(r.sums, 2), (mass[tt], energy[tt])), tt
    for k in FIELDS:
        assert np.array_equal(st.download(k), sa.download(k)), k
    b.free()
    for s, x in ((sa, ma), (st, m)):
        s.close()
        x.close()
