"""Workloads of the hydro kernel set, as programs that use it run them.

A pass is a whole solve: the initial density, energy and (zero) momenta are put
back into the device arrays, the driver loop runs for some steps, and the
carried fields, the mass fluxes, the dt sequence and the totals come back.

kinds
  run        the driver loop in C: flowhip_run (FP64) or flowhip_run_f32
  interface  the same loop in the caller, one solve_hydro_2d and one
             print_conservation call per step, as flow's own main.c drives it
  ensemble   many meshes of uneven sizes advanced together, graphs on
"""
import ctypes
import math
import random

import numpy as np
import torch

import flow_amd

GAMMA, C_Q, C_T = 1.4, 3.0, 0.3
PAD = 2
FIELDS = ("rho", "e", "u", "v", "mom_x", "mom_y")
FLUXES = ("F_x", "F_y")
ZEROS = ("mom_x", "mom_y", "Qxx", "Qyy")  # zero in an initial state


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------

def _single(name, kind, fp32, nx, ny, steps, problem):
    return {"name": name, "kind": kind, "fp32": fp32, "nx": nx, "ny": ny, "steps": steps,
            "problem": problem}


def _ensemble(name, fp32, count, lo, hi, steps, autotune):
    return {"name": name, "kind": "ensemble", "fp32": fp32, "count": count, "lo": lo,
            "hi": hi, "steps": steps, "autotune": autotune}


def listed():
    return [
        # a quick look at a problem: every step is launches and latency
        _single("run_64", "run", False, 64, 64, 50, "split"),
        # the 512^2 shock tube, the smallest of the benchmark's configurations
        _single("run_512", "run", False, 512, 512, 50, "split"),
        # an ordinary size that is not a power of two
        _single("run_1000", "run", False, 1000, 1000, 30, "box"),
        # a channel: long rows, few of them, both sides ragged
        _single("run_3000x150", "run", False, 3000, 150, 30, "split"),
        # odd sides, larger than the caches
        _single("run_3001x2999", "run", False, 3001, 2999, 10, "blasts"),
        # the size of flow.params, driven through the two interface calls
        _single("interface_4096", "interface", False, 4096, 4096, 10, "box"),
        # the benchmark's roofline configuration
        _single("run_8192", "run", False, 8192, 8192, 8, "blasts"),
        # the FP32-state form: small, ordinary (not a power of two), largest
        _single("f32_300x200", "run", True, 300, 200, 50, "split"),
        _single("f32_1536", "run", True, 1536, 1536, 20, "blasts"),
        _single("f32_8192", "run", True, 8192, 8192, 8, "blasts"),
        # a parameter study of small meshes, schedule as it comes
        _ensemble("ensemble_24", False, 24, 64, 512, 40, False),
        # the batching benchmark's range of sides, autotuned first
        _ensemble("ensemble_f32_96", True, 96, 64, 1024, 20, True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    what = rng.random()
    fp32 = rng.random() < 0.4
    if what < 0.2:
        count = _log_int(rng, 8, 96)
        hi = _log_int(rng, 200, 1024)
        return {k: v for k, v in _ensemble("", fp32, count, 64, hi, rng.randint(12, 24),
                                           rng.random() < 0.5).items() if k != "name"}
    nx = _log_int(rng, 40, 8192)
    # square half of the time, else up to a factor of 12 from it
    ny = nx if rng.random() < 0.5 else max(24, min(8192, int(nx * math.exp(rng.uniform(-2.5, 2.5)))))
    steps = max(6, min(50, int(3.0e8 / (nx * ny))))
    kind = "interface" if what < 0.4 and not fp32 else "run"
    problem = rng.choice(["split", "box", "blasts"])
    return {k: v for k, v in _single("", kind, fp32, nx, ny, steps, problem).items()
            if k != "name"}


def _members(case):
    """The sides of an ensemble's instances, the same for every seed."""
    rng = random.Random("sides %d %d %d" % (case["count"], case["lo"], case["hi"]))
    return [_log_int(rng, case["lo"], case["hi"]) for _ in range(case["count"])]


def work(case):
    """Per cell and step: density, energy and the two momenta read once, the
    six carried fields written once. The operations are those of the step's
    expressions (quotients and roots counted as one)."""
    if case["kind"] == "ensemble":
        cells = sum(n * n for n in _members(case))
    else:
        cells = case["nx"] * case["ny"]
    size = 4 if case["fp32"] else 8
    return {"bytes": 10.0 * size * cells * case["steps"], "flops": 380.0 * cells * case["steps"]}


# --------------------------------------------------------------------------
# initial states: made on the GPU from the seed
# --------------------------------------------------------------------------

def _initial(nx, ny, problem, seed):
    """(rho, e, dt): padded (ny+4, nx+4) float64 tensors with reflected
    ghosts (corners zero), and a .params dt below the CFL limit."""
    rng = random.Random("state %d" % seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    x = (torch.arange(nx, device="cuda", dtype=torch.float64) + 0.5) / nx
    y = (torch.arange(ny, device="cuda", dtype=torch.float64) + 0.5) / ny
    rho = torch.empty(ny, nx, device="cuda", dtype=torch.float64)
    p = torch.empty_like(rho)
    if problem == "split":       # a Sod-type shock tube
        at = rng.uniform(0.3, 0.7)
        p_hi = 0.1 * math.exp(rng.uniform(math.log(10.0), math.log(100.0)))
        left = (x < at)[None, :].expand(ny, nx)
        rho.copy_(torch.where(left, 1.0, 0.125))
        p.copy_(torch.where(left, p_hi, 0.1))
    elif problem == "box":       # flow.params' dense box in a thin gas
        side, p_hi = rng.uniform(0.1, 0.3), rng.uniform(0.8, 1.2)
        inside = ((x - 0.5).abs() < side)[None, :] & ((y - 0.5).abs() < side)[:, None]
        rho.copy_(torch.where(inside, 1.0, 0.125))
        p.copy_(torch.where(inside, p_hi, 0.1))
    else:                        # a 4 x 4 grid of blasts
        rho.fill_(1.0)
        p.fill_(0.1)
        p_hi = 0.0
        for l in range(4):
            for k in range(4):
                pk = math.exp(rng.uniform(math.log(10.0), math.log(1000.0)))
                p_hi = max(p_hi, pk)
                inside = (((x - (k + 0.5) / 4).abs() < 0.025)[None, :] &
                          ((y - (l + 0.5) / 4).abs() < 0.025)[:, None])
                p.masked_fill_(inside, pk)
    noise = torch.rand(ny, nx, device="cuda", dtype=torch.float64, generator=gen)
    rho.mul_(1.0 + 0.05 * (2.0 * noise - 1.0))
    e = p / ((GAMMA - 1.0) * rho)
    fastest = math.sqrt(GAMMA * p_hi / 0.95)
    dt = 0.2 * min(1.0 / nx, 1.0 / ny) / fastest
    out = []
    for a in (rho, e):
        full = torch.zeros(ny + 2 * PAD, nx + 2 * PAD, device="cuda", dtype=torch.float64)
        full[PAD:-PAD, PAD:-PAD] = a
        out.append(_reflect(full))
    return out[0], out[1], dt


def _reflect(a, sx=1.0, sy=1.0):
    """The pad-2 reflective boundary, in place: mirrored rows and columns,
    corners untouched; sx negates the columns, sy the rows."""
    c = slice(PAD, -PAD)
    a[1, c], a[0, c] = sy * a[2, c], sy * a[3, c]
    a[-2, c], a[-1, c] = sy * a[-3, c], sy * a[-4, c]
    a[c, 1], a[c, 0] = sx * a[c, 2], sx * a[c, 3]
    a[c, -2], a[c, -1] = sx * a[c, -3], sx * a[c, -4]
    return a


# --------------------------------------------------------------------------
# what a program holds, and one pass
# --------------------------------------------------------------------------

class _Device:
    """A device array of the kernel set, for torch.as_tensor. Its tensors keep
    it, and with it the owner that frees the memory, alive."""

    def __init__(self, owner, ptr, count, fp32):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "data": (int(ptr), False),
                                         "typestr": "<f4" if fp32 else "<f8", "version": 2}


def _tensor(owner, ptr, count, fp32):
    return torch.as_tensor(_Device(owner, ptr, count, fp32), device="cuda")


def _flat(a, count, fp32):
    """A padded 2-D array as the kernel set lays it out, `count` values."""
    full = torch.zeros(count, device="cuda", dtype=torch.float32 if fp32 else torch.float64)
    full[: a.numel()] = a.reshape(-1)
    return full


class _Solve:
    pass


def prepare(case, seed):
    if case["kind"] == "ensemble":
        return _prepare_ensemble(case, seed)
    s = _Solve()
    s.case, fp32 = case, case["fp32"]
    nx, ny = case["nx"], case["ny"]
    rho, e, s.dt = _initial(nx, ny, case["problem"], seed)
    s.mesh = flow_amd.Mesh(nx, ny, dt=s.dt)
    s.device = flow_amd.DeviceState32(s.mesh) if fp32 else flow_amd.DeviceState(s.mesh)
    s.fields = {k: _tensor(s.device, s.device.ptrs[k], s.device.n, fp32) for k in FIELDS + FLUXES}
    s.zeros = [_tensor(s.device, s.device.ptrs[k], s.device.n, fp32) for k in ZEROS]
    s.rho, s.e = _flat(rho, s.device.n, fp32), _flat(e, s.device.n, fp32)
    torch.cuda.synchronize()
    return s


def _prepare_ensemble(case, seed):
    s = _Solve()
    s.case, fp32 = case, case["fp32"]
    sides = _members(case)
    states = [_initial(n, n, ("split", "box", "blasts")[k % 3], seed * 1000 + k)
              for k, n in enumerate(sides)]
    s.dt = [st[2] for st in states]
    s.ens = flow_amd.Ensemble(sides, dt=min(s.dt), fp32=fp32)
    s.rho, s.e = [], []
    arrays = {k: [] for k in FIELDS + ZEROS}
    for k, n in enumerate(sides):
        count = (n + 5) * (n + 5)
        for name, found in arrays.items():
            ptr = flow_amd.lib().flowhip_ensemble_array(
                s.ens.ptr, k, flow_amd.ARRAY_NAMES.index(name))
            found.append(_tensor(s.ens, ptr, count, fp32))
        s.rho.append(_flat(states[k][0], count, fp32))
        s.e.append(_flat(states[k][1], count, fp32))
    s.fields = {k: arrays[k] for k in FIELDS}
    s.zeros = [a for k in ZEROS for a in arrays[k]]
    _put_back(s)
    if case["autotune"]:
        s.ens.autotune(trial_steps=3)
    s.ens.set_graphs(True)
    torch.cuda.synchronize()
    return s


def _put_back(s):
    """The initial state, into the kernel set's arrays. The solve works on a
    stream of its own, so what torch wrote has to be there first."""
    if s.case["kind"] == "ensemble":
        torch._foreach_copy_(s.fields["rho"], s.rho)
        torch._foreach_copy_(s.fields["e"], s.e)
        torch._foreach_zero_(s.zeros)
        for k, dt in enumerate(s.dt):
            flow_amd.lib().flowhip_ensemble_set_dt(s.ens.ptr, k, C_T * dt, C_T * dt)
    else:
        s.fields["rho"].copy_(s.rho)
        s.fields["e"].copy_(s.e)
        torch._foreach_zero_(s.zeros)
        s.mesh.set_dt(C_T * s.dt, C_T * s.dt)
    torch.cuda.current_stream().synchronize()


def run(s):
    case = s.case
    steps = case["steps"]
    _put_back(s)
    if case["kind"] == "ensemble":
        dts, mass, energy, _ = s.ens.run(steps)
        out = {k: torch.cat(s.fields[k]) for k in FIELDS}
        out.update(dt=dts, mass=mass, energy=energy)
        return out
    if case["kind"] == "run":
        _, dts, mass, energy, _ = s.device.run(steps)
        out = dict(s.fields)
        out.update(dt=dts, mass=mass, energy=energy)
        return out
    lib, mesh, dev = flow_amd.lib(), s.mesh, s.device
    dev.set_timestep(0)
    dts = [(mesh.dt, mesh.dt_h)]
    for tt in range(steps):
        dev.solve(tt)
        lib.print_conservation(mesh.nx, mesh.ny, ctypes.c_void_p(dev.ptrs["rho"]),
                               ctypes.c_void_p(dev.ptrs["e"]), None, mesh.ptr)
        dts.append((mesh.dt, mesh.dt_h))
    out = dict(s.fields)
    out.update(dt=np.array(dts))
    return out


# --------------------------------------------------------------------------
# the same solve in 64 bits, in plain torch
# --------------------------------------------------------------------------
# Arrays are (rows, columns) with two ghosts on each side: cells (Ly, Lx),
# x faces (Ly, Lx+1), y faces (Ly+1, Lx). Sweeps are written along the last
# axis; the y sweeps pass transposed views.

def _minmod(a, b):
    return torch.where(a * b > 0, torch.where(a.abs() < b.abs(), a, b), 0.0)


def _ratio(a, b):
    return torch.where(b == 0, 0.0, a / torch.where(b == 0, 1.0, b))


def _sh(a, lo, n):
    """n entries of the last axis from position lo."""
    return a[..., lo:lo + n]


def _between(w0, w1, w2, w3, low, vel, d, dt_h):
    """Monotonised-central value between w1 and w2, upwind of vel."""
    def slope(p, q, r):
        return _minmod(_minmod(0.5 / d * (r - p), 2.0 / d * (q - p)), 2.0 / d * (r - q))
    return torch.where(low, w1 + 0.5 * slope(w0, w1, w2) * (d - vel * dt_h),
                       w2 - 0.5 * slope(w1, w2, w3) * (d + vel * dt_h))


def _face_flux(vel, rho, e, d, across, dt, dt_h, sel_by_face):
    """Mass and energy flux at the faces [2, L-2] of the last axis; vel lives
    on faces (L+1), rho and e on cells (L). Rows as given."""
    n = rho.shape[-1] - 3
    v0, vm, vp = _sh(vel, 2, n), _sh(vel, 1, n), _sh(vel, 3, n)
    r = [_sh(rho, k, n) for k in range(4)]
    q = [_sh(e, k, n) for k in range(4)]
    v = v0 - 0.5 * v0 * dt * _minmod(0.5 / d * (vp - vm),
                                     _minmod(2.0 / d * (v0 - vm), 2.0 / d * (vp - v0)))
    jump = r[2] - r[1]
    sel = v0 if sel_by_face else v
    smooth = _ratio(torch.where(sel >= 0, r[1] - r[0], r[3] - r[2]), jump)
    limiter = torch.where(jump == 0, 0.0, (smooth + smooth.abs()) / (1.0 + smooth.abs()))
    mass = (v * torch.where(v >= 0, r[1], r[2]) +
            0.5 * v.abs() * (1.0 - (v * dt_h / d).abs()) * limiter * jump)
    return mass, across * _between(*q, v > 0, v, d, dt_h) * mass


def _sweep(vel, rho, rho_old, e, flux, d, across, dt, dt_h, first, sel_by_face):
    """One directional sweep along the last axis, interior rows only; flux
    (faces) is written, and the new rho and e are returned (ghosts stale)."""
    c = slice(PAD, -PAD)
    mass, energy = _face_flux(vel[c], rho[c], e[c], d, across, dt, dt_h, sel_by_face)
    flux[c, PAD:-PAD] = mass
    rho, e, area = rho.clone(), e.clone(), d * across
    old = rho_old[c, c]
    rho_e = old * e[c, c] - dt_h * (energy[:, 1:] - energy[:, :-1]) / area
    rho[c, c] = rho[c, c] - dt_h * (across * mass[:, 1:] - across * mass[:, :-1]) / area
    e[c, c] = _ratio(rho_e, old if first else rho[c, c])
    return rho, e


def _edge(rho):
    """Densities at the faces [2, L-2] of the last axis."""
    return 0.5 * (rho[..., 2:-1] + rho[..., 1:-2])


def _along(w, f, d, across, dt_h):
    """Flux at cells [2, L-2) of the velocity w on faces of the last axis,
    carried by the mass flux f."""
    n = w.shape[-1] - 5
    vel = 0.5 * (_sh(w, 2, n) + _sh(w, 3, n))
    return (across * 0.5 * (_sh(f, 2, n) + _sh(f, 3, n)) *
            _between(_sh(w, 1, n), _sh(w, 2, n), _sh(w, 3, n), _sh(w, 4, n), vel > 0, vel, d,
                     dt_h))


def _across(w, carrier, f, d, across, dt_h):
    """Flux at the faces [2, L-2] of the last axis of w (which has L entries
    there), carried by `carrier` and f, given averaged at those points."""
    n = w.shape[-1] - 3
    return (across * f * _between(_sh(w, 0, n), _sh(w, 1, n), _sh(w, 2, n), _sh(w, 3, n),
                                  carrier > 0, carrier, d, dt_h))


def _momentum(own, other, mom, rho, f_own, f_other, d, b, dt_h, along_first):
    """Advection of the momentum along the last axis; `own` is its velocity
    (rows: cells, columns: faces), `other` the velocity of the row axis (rows:
    faces, columns: cells), f_* the mass fluxes of the same layouts; d, b the
    spacings of the last axis and of the rows. Returns the new velocity."""
    c, n = slice(PAD, -PAD), own.shape[-1] - 4
    faces = slice(PAD, PAD + n)
    # at corners (rows: row faces, columns: own faces)
    carrier = 0.5 * (other[c, 1:-2] + other[c, 2:-1])
    f_corner = 0.5 * (f_other[c, 1:-2] + f_other[c, 2:-1])

    def flux_along(w):  # cells [1, L-1) of the row: the flux mirrored into the ghosts
        g = _along(w[c], f_own[c], d, b, dt_h)
        g = torch.cat([g[:, :1], g, g[:, -1:]], 1)
        return (g[:, 1:] - g[:, :-1]) / (d * b)

    def flux_across(w):
        g = _across(w[:, faces].T, carrier.T, f_corner.T, b, d, dt_h).T
        return (g[1:] - g[:-1]) / (d * b)

    order = (flux_along, flux_across) if along_first else (flux_across, flux_along)
    mom[c, faces] -= dt_h * order[0](own)
    own = own.clone()
    own[c, faces] = _ratio(mom[c, faces], _edge(rho[c]))
    _reflect(own, sx=-1.0)
    mom[c, faces] -= dt_h * order[1](own)
    return own


def _timestep(rho, e, qx, qy, dx, dy, dt_h, first):
    c = slice(PAD, -PAD)
    c2 = GAMMA * (GAMMA - 1.0) * e[c, c]
    dtx = dx / (c2 + 2.0 * qx[c, c] / rho[c, c]).sqrt()
    dty = dy / (c2 + 2.0 * qy[c, c] / rho[c, c]).sqrt()
    low = torch.minimum(dtx, dty)
    low = torch.where(low.isnan(), math.inf, low).min().item()
    low = min(1.0e30, low, 1.5 / C_T * dt_h)
    dt = 0.5 * (C_T * low + dt_h)
    return dt, (dt if first else C_T * low)


def _stress(w, rho):
    """Viscous stress of the cells [2, L-2) along the last axis."""
    step = (w[..., 1:] - w[..., :-1]).clamp(max=0.0)
    n = rho.shape[-1] - 4
    m, z, p = _sh(step, 1, n), _sh(step, 2, n), _sh(step, 3, n)
    return -C_Q * rho[..., PAD:-PAD] * z * (0.5 * ((p - z).abs() + (z - m).abs()))


def _exact_solve(rho, e, dt, steps):
    Ly, Lx = rho.shape
    dx, dy = 1.0 / (Lx - 2 * PAD), 1.0 / (Ly - 2 * PAD)
    c = slice(PAD, -PAD)
    like = dict(device=rho.device, dtype=torch.float64)
    mx, F_x = torch.zeros(Ly, Lx + 1, **like), torch.zeros(Ly, Lx + 1, **like)
    my, F_y = torch.zeros(Ly + 1, Lx, **like), torch.zeros(Ly + 1, Lx, **like)
    u, v = torch.zeros_like(mx), torch.zeros_like(my)
    qx, qy = torch.zeros_like(rho), torch.zeros_like(rho)
    dt = dt_h = C_T * dt
    dt, dt_h = _timestep(rho, e, qx, qy, dx, dy, dt_h, False)
    pairs, mass, energy = [(dt, dt_h)], [], []

    def accelerate(mom, vel, a, density, d):
        mom[c, c] -= dt * (a[:, 2:-1] - a[:, 1:-2])[c] / d
        vel[c, c] = _ratio(mom[c, c], _edge(density[c]))
        _reflect(vel, sx=-1.0)

    for tt in range(steps):
        P = (GAMMA - 1.0) * rho * e
        # views of the y fields with their axes exchanged: the same code
        accelerate(mx, u, P, rho, dx)
        accelerate(my.T, v.T, P.T, rho.T, dy)
        qx[c, c], qy[c, c] = _stress(u[c], rho[c]), _stress(v.T[c], rho.T[c]).T
        _reflect(qx), _reflect(qy)
        accelerate(mx, u, qx, rho, dx)
        accelerate(my.T, v.T, qy.T, rho.T, dy)

        dvx = (u[c, 3:-2] - u[c, 2:-3]) / dx
        dvy = (v[3:-2, c] - v[2:-3, c]) / dy
        div = (dvx + dvy) * dt_h
        r, p, e0 = rho[c, c], P[c, c], e[c, c]
        e_q = e0 - dt_h * (qx[c, c] * dvx + qy[c, c] * dvy) / r
        e_c = e_q - p * div / r
        work_done = 0.5 * div * (p + (GAMMA - 1.0) * e_c * (r / (1.0 + div))) / r
        e[c, c] = torch.where(r == 0, 0.0, e_q - work_done)
        _reflect(e)
        dt, dt_h = _timestep(rho, e, qx, qy, dx, dy, dt_h, tt == 0)

        old = rho.clone()
        for k in range(2):
            first = k == 0
            if (tt % 2 == 0) == first:
                rho, e = _sweep(u, rho, old, e, F_x, dx, dy, dt, dt_h, first, False)
                _reflect(F_x, sx=-1.0)
            else:
                rt, et = _sweep(v.T, rho.T, old.T, e.T, F_y.T, dy, dx, dt, dt_h, first, True)
                rho, e = rt.T.contiguous(), et.T.contiguous()
                _reflect(F_y, sy=-1.0)
            _reflect(rho), _reflect(e)
        u = _momentum(u, v, mx, rho, F_x, F_y, dx, dy, dt_h, tt % 2 == 1)
        v = _momentum(v.T, u.T, my.T, rho.T, F_y.T, F_x.T, dy, dx, dt_h,
                      tt % 2 == 0).T.contiguous()
        pairs.append((dt, dt_h))
        mass.append(rho[c, c].sum().item())
        energy.append((rho[c, c] * e[c, c]).sum().item())
    fields = {"rho": rho, "e": e, "u": u, "v": v, "mom_x": mx, "mom_y": my, "F_x": F_x,
              "F_y": F_y}
    return fields, np.array(pairs), np.array(mass), np.array(energy)


def exact(case, seed):
    if case["kind"] == "ensemble":
        sides, got = _members(case), []
        if case["count"] * case["steps"] > 2400:
            return None  # thousands of small steps: too long one by one
        for k, n in enumerate(sides):
            rho, e, dt = _initial(n, n, ("split", "box", "blasts")[k % 3], seed * 1000 + k)
            f, pairs, mass, energy = _exact_solve(rho, e, dt, case["steps"])
            got.append(({q: _flat(f[q], (n + 5) * (n + 5), False) for q in FIELDS}, pairs,
                        mass, energy))
        out = {q: torch.cat([g[0][q] for g in got]) for q in FIELDS}
        out.update(dt=np.stack([g[1] for g in got]), mass=np.stack([g[2] for g in got]),
                   energy=np.stack([g[3] for g in got]))
        return out
    rho, e, dt = _initial(case["nx"], case["ny"], case["problem"], seed)
    count = (case["nx"] + 5) * (case["ny"] + 5)
    f, pairs, mass, energy = _exact_solve(rho, e, dt, case["steps"])
    out = {k: _flat(f[k], count, False) for k in FIELDS + FLUXES}
    out.update(dt=pairs)
    if case["kind"] == "run":
        out.update(mass=mass, energy=energy)
    return out
