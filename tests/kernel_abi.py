"""ctypes mirrors of flow_hip_kernels.h's structs, for tests that call the
kernel launchers themselves."""
import ctypes

from flow_amd import native

_vp, _i, _d = ctypes.c_void_p, ctypes.c_int, ctypes.c_double
QUEUE_WORDS = 768


class FkUniform(ctypes.Structure):
    _fields_ = [(k, _d) for k in ("edx", "edy", "cdx", "cdy", "iedx", "iedy", "rcdx", "rcdy")]


class FkMesh(ctypes.Structure):
    """FkMesh, and FkMesh32 (the same layout)."""
    _fields_ = ([(k, _i) for k in ("nx", "ny", "pad")] +
                [(k, _vp) for k in ("edgedx", "edgedy", "celldx", "celldy", "inv_edgedx",
                                    "inv_edgedy")] +
                [("pow2", _i), ("uniform", _i), ("u", FkUniform), ("pairs", _i)])


class FkReduce(ctypes.Structure):
    _fields_ = [(k, _vp) for k in ("partials", "dtp", "sums", "status", "queue", "mail", "cfl")]


def lib():
    L = ctypes.CDLL(native.library_path())
    for suffix in ("", "_f32"):
        for name, args in (
                ("fk_march_lagrangian", [FkMesh] + [_vp] * 10 + [FkReduce, _d, _vp, _i, _vp]),
                ("fk_march_mass_energy",
                 [FkMesh, _i] + [_vp] * 8 + [FkReduce, _d, _i, _i, _vp, _i, _vp]),
                ("fk_march_momentum",
                 [FkMesh, _i] + [_vp] * 11 + [FkReduce, _i, _i, _vp]),
                ("fk_march_momentum_x", [FkMesh, _i] + [_vp] * 8 + [FkReduce, _i, _vp]),
                ("fk_march_momentum_y", [FkMesh, _i] + [_vp] * 8 + [FkReduce, _i, _i, _vp])):
            fn = getattr(L, name + suffix)
            fn.restype, fn.argtypes = _i, args
    return L


def mesh(fp32, nx, ny, pairs=0):
    """A mesh of uniform spacings 1/64, by value only."""
    u = FkUniform(*([1.0 / 64] * 4 + [64.0] * 4))
    return FkMesh(nx=nx, ny=ny, pad=2, pow2=1, uniform=1, u=u, pairs=pairs)


def march_calls(L, m, fp32, tt, rows):
    """The results of the march launchers of a step with no arrays."""
    suffix = "_f32" if fp32 else ""
    r = FkReduce(queue=256)
    parts = ctypes.c_int()
    out = [getattr(L, "fk_march_lagrangian" + suffix)(m, *[None] * 10, r, 1.0,
                                                      ctypes.byref(parts), rows, None),
           getattr(L, "fk_march_mass_energy" + suffix)(m, tt, *[None] * 8, r, 1.0, 0, 1,
                                                       ctypes.byref(parts), rows, None),
           getattr(L, "fk_march_momentum" + suffix)(m, tt, *[None] * 11, r, 1, rows, None),
           getattr(L, "fk_march_momentum_x" + suffix)(m, tt, *[None] * 8, r, rows, None),
           getattr(L, "fk_march_momentum_y" + suffix)(m, tt, *[None] * 8, r, 1, rows, None)]
    return out
