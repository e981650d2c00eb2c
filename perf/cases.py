"""Performance cases of the GPU path: what one time step of a MDOODZ run asks
of this library, through its public entry points, with every array resident
in device memory (as PicardLoop(device=True) and bench.py keep them).

  markers   mdg_markers_set on the moved markers, then P2Mastah_Fused of four
            fields onto the centres and three onto the vertices and the phase
            fractions: the marker -> grid half of a step.
  advect    pressure and stress increments onto the markers, then the RK4
            advection: the grid -> marker half of a step.
  rheology  one evaluation of the non-linear residual (strain rates, node
            averages, viscosity on centres and vertices, residual), with the
            tangent coefficients of a Newton step where "newton" is set.
  solve     the linear Stokes solve (KillerSolver's replacement).
  energy    the implicit energy step (Jacobi PCG).
  network   the learned preconditioner: forward pass, or loss and gradient.

torch is imported before the library, so that both use one HIP runtime;
torch tensors view the library's device arrays without copies."""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mdoodz7.0_amd"))

import mdgpu  # noqa: E402
from mdgpu import learned  # noqa: E402
from mdgpu import setups as S  # noqa: E402

F64 = torch.float64
# the solver options that bench.py measures (vertex-patch smoother), FP64 and
# FP32 V-cycle
PATCH = dict(smoother=3, penalty=700.0, cheb_degree=12, cheb_degree_coarse=12)
PATCH_MIXED = dict(PATCH, penalty=300.0, precision=mdgpu.MDG_PREC_MIXED)
LAYERS = learned.LAYERS


def listed():
    return [
        # the 101^2 inclusion set-up, 16 markers a cell: launch latency
        dict(name="markers_101", kind="markers", nx=101, nz=101, per=4, stencil=1, phases=2, stirred=False),
        # a ragged box with the 9-cell stencil, markers moved by a flow
        dict(name="markers_637x301_s9", kind="markers", nx=637, nz=301, per=3, stencil=9, phases=4, stirred=True),
        # the 2047^2 workload's 37.7M markers after some time steps
        dict(name="markers_2047", kind="markers", nx=2047, nz=2047, per=3, stencil=1, phases=9, stirred=True),
        # a small ragged box, plain bilinear velocities
        dict(name="advect_255x127", kind="advect", nx=255, nz=127, per=4, conserv=0),
        # 37.7M markers with the conservative velocity interpolation
        dict(name="advect_2047", kind="advect", nx=2047, nz=2047, per=3, conserv=1),
        # the shear-band box: power law, Maxwell, Drucker-Prager
        dict(name="rheology_1023_vep", kind="rheology", nx=1023, nz=1023, law="vep", newton=False),
        # a quarter of the 4095 x 1023 lithosphere: dislocation, diffusion
        # and Peierls creep in three layers, with the Newton tangent
        dict(name="rheology_1023x255_creep", kind="rheology", nx=1023, nz=255, law="creep", newton=True),
        # the 101^2 inclusion under pure shear with the default options
        dict(name="solve_101", kind="solve", nx=101, nz=101, body="inclusion", opts="default"),
        # ellipses with a contrast of 1e6, the tuned FP64 solver
        dict(name="solve_383_fp64", kind="solve", nx=383, nz=383, body="ellipses", opts="patch"),
        # the same kind of field at 767^2 with the FP32 V-cycle
        dict(name="solve_767_mixed", kind="solve", nx=767, nz=767, body="ellipses", opts="patch_mixed"),
        # the energy step on the 2047^2 grid
        dict(name="energy_2047", kind="energy", nx=2047, nz=2047, fourier=32.0),
        # one training gradient of the network at its training size
        dict(name="network_grad_256", kind="network", h=256, w=256, grad=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over the ranges that the listed cases span."""
    kind = rng.choice(["markers", "advect", "rheology", "solve", "energy", "network"])
    if kind in ("markers", "advect"):
        nx, nz = _log_int(rng, 60, 1800), _log_int(rng, 60, 1800)
        per = rng.choice([3, 4])
        if kind == "markers":
            s = rng.choice([1, 1, 9])
            if s == 9:      # the 9-cell stencil reads each marker several times
                nx, nz = min(nx, 700), min(nz, 700)
            return dict(kind=kind, nx=nx, nz=nz, per=per, stencil=s, phases=rng.randint(2, 9),
                        stirred=rng.random() < 0.7)
        return dict(kind=kind, nx=nx, nz=nz, per=per, conserv=rng.randint(0, 1))
    if kind == "rheology":
        law = rng.choice(["vep", "creep"])
        return dict(kind=kind, nx=_log_int(rng, 60, 1000), nz=_log_int(rng, 60, 500), law=law,
                    newton=rng.random() < 0.4)
    if kind == "solve":
        if rng.random() < 0.4:
            return dict(kind=kind, nx=_log_int(rng, 40, 140), nz=_log_int(rng, 40, 140), body="inclusion",
                        opts=rng.choice(["default", "patch"]))
        n = _log_int(rng, 100, 360)
        return dict(kind=kind, nx=n, nz=max(64, int(n * rng.uniform(0.7, 1.0))), body="ellipses",
                    opts=rng.choice(["patch", "patch_mixed"]))
    if kind == "energy":
        return dict(kind=kind, nx=_log_int(rng, 60, 2000), nz=_log_int(rng, 60, 2000),
                    fourier=round(math.exp(rng.uniform(0.0, math.log(40.0))), 2))
    return dict(kind=kind, h=8 * _log_int(rng, 8, 96), w=8 * _log_int(rng, 8, 96), grad=rng.random() < 0.6)


# ------------------------------------------------------------ device arrays
class _Span:
    """__cuda_array_interface__ of a DeviceArray (kept alive by the tensor)."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = dict(shape=(a.n,), typestr=np.dtype(a.dtype).str, data=(a.p, False),
                                             version=2, strides=None)


def _tensor(a):
    """A torch view of a DeviceArray."""
    return torch.as_tensor(_Span(a), device="cuda")


def _upload(ctx, t):
    """A DeviceArray with the values of a torch tensor."""
    t = t.contiguous()
    dt = {torch.float64: np.float64, torch.float32: np.float32, torch.int32: np.int32, torch.int8: np.int8}[t.dtype]
    a = ctx.device(t.numel(), dt)
    _tensor(a).copy_(t.reshape(-1))
    return a


def _zeros(ctx, n):
    return _upload(ctx, torch.zeros(n, dtype=F64, device="cuda"))


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _uniform(gen, n, lo, hi):
    return torch.rand(n, dtype=F64, device="cuda", generator=gen) * (hi - lo) + lo


def _closed_box(nx, nz):
    """Boundary tags of a closed free-slip box of nx x nz cells."""
    Nx, Nz = nx + 1, nz + 1
    tu = np.full((Nz + 1, Nx), -1, np.int8)
    tu[:, 0] = tu[:, -1] = 0
    tu[0] = tu[-1] = 13
    tv = np.full((Nz, Nx + 1), -1, np.int8)
    tv[0] = tv[-1] = 0
    tv[:, 0] = tv[:, -1] = 13
    return (tu.ravel(), np.zeros(tu.size), tv.ravel(), np.zeros(tv.size), np.full(nx * nz, -1, np.int8),
            np.full(Nx * Nz, -1, np.int8))


def _box(case):
    """Cells of equal width and height: the longer side is 1."""
    m = max(case["nx"], case["nz"])
    return 0.0, case["nx"] / m, 0.0, case["nz"] / m


def _context(case):
    c = mdgpu.Context(case["nx"] + 1, case["nz"] + 1, *_box(case))
    c.set_bc(*_closed_box(case["nx"], case["nz"]))
    return c


def _coords(case):
    x0, x1, z0, z1 = _box(case)
    g = S.grid_coords(case["nx"] + 1, case["nz"] + 1, x0, x1, z0, z1)
    return {k: torch.as_tensor(v, device="cuda") if isinstance(v, np.ndarray) else v for k, v in g.items()}


# ------------------------------------------------------------------ markers
def _turn(x, z, Lx, Lz, T, steps):
    """Positions after time T in the cellular flow of one vortex."""
    def vel(a, b):
        return (torch.sin(math.pi * a / Lx) * torch.cos(math.pi * b / Lz),
                -torch.cos(math.pi * a / Lx) * torch.sin(math.pi * b / Lz) * (Lz / Lx))
    h = T / steps
    for _ in range(steps):
        a, b = vel(x, z)
        a, b = vel(x + 0.5 * h * a, z + 0.5 * h * b)
        x, z = x + h * a, z + h * b
    return x.clamp(1e-9 * Lx, Lx * (1 - 1e-9)), z.clamp(1e-9 * Lz, Lz * (1 - 1e-9))


def _positions(case, gen, stirred):
    """Markers in the order that MDOODZ places them (cell column outer, cell
    row inner) with a jitter; "stirred" ones have since moved with a flow."""
    nx, nz, per = case["nx"], case["nz"], case["per"]
    x0, x1, z0, z1 = _box(case)
    dx, dz = (x1 - x0) / nx, (z1 - z0) / nz
    sub = (torch.arange(per, dtype=F64, device="cuda") + 0.5) / per
    gx = (torch.arange(nx, dtype=F64, device="cuda")[:, None, None, None] + sub[None, None, :, None]) * dx
    gz = (torch.arange(nz, dtype=F64, device="cuda")[None, :, None, None] + sub[None, None, None, :]) * dz
    shape = (nx, nz, per, per)
    x, z = gx.expand(shape).reshape(-1), gz.expand(shape).reshape(-1)
    n = x.numel()
    x = x + _uniform(gen, n, -0.1, 0.1) * (dx / per)
    z = z + _uniform(gen, n, -0.1, 0.1) * (dz / per)
    if stirred:
        x, z = _turn(x, z, x1, z1, 0.6, 24)
    return x, z


def _phases(x, z, case, gen, nph):
    """Random ellipses of nph - 1 materials in a matrix."""
    x0, x1, z0, z1 = _box(case)
    m = 24
    p = torch.rand((m, 6), dtype=F64, device="cuda", generator=gen).cpu().numpy()
    ph = torch.zeros(x.numel(), dtype=torch.int32, device="cuda")
    for i in range(m):
        c, s = math.cos(math.pi * p[i, 4]), math.sin(math.pi * p[i, 4])
        xr, zr = x - x1 * p[i, 0], z - z1 * p[i, 1]
        a, b = 0.03 + 0.08 * p[i, 2], 0.03 + 0.08 * p[i, 3]
        ph[((c * xr + s * zr) / a) ** 2 + ((c * zr - s * xr) / b) ** 2 <= 1.0] = 1 + i % (nph - 1)
    return ph


def _tables(case):
    k = np.arange(case["phases"])
    return 10.0 ** (3.0 * np.sin(1.0 + 2.0 * k)), 2700.0 + 75.0 * k, 1e10 * (1.0 + 0.3 * k)


def _markers_inputs(case, seed):
    gen = _gen(seed)
    x, z = _positions(case, gen, case["stirred"])
    ph = _phases(x, z, case, gen, case["phases"])
    T = 600.0 + 700.0 * z + _uniform(gen, x.numel(), -20.0, 20.0)
    return x, z, ph, T


def _prepare_markers(case, seed):
    x, z, ph, T = _markers_inputs(case, seed)
    c = _context(case)
    st = dict(ctx=c, x=_upload(c, x), z=_upload(c, z), ph=_upload(c, ph), T=_upload(c, T), stencil=case["stencil"],
              nph=case["phases"])
    nc, nv = c.node_count(1), c.node_count(0)
    eta, rho, G = _tables(case)
    st["cent"] = [dict(src=eta, dst=_zeros(c, nc), flag=0, avg=2), dict(src=rho, dst=_zeros(c, nc), flag=0, avg=0),
                  dict(src=G, dst=_zeros(c, nc), flag=0, avg=1), dict(src=st["T"], dst=_zeros(c, nc), flag=1, avg=0)]
    st["vert"] = [dict(src=eta, dst=_zeros(c, nv), flag=0, avg=2), dict(src=rho, dst=_zeros(c, nv), flag=0, avg=0),
                  dict(src=G, dst=_zeros(c, nv), flag=0, avg=1)]
    st["perc"] = [_zeros(c, nc) for _ in range(case["phases"])]
    st["none"] = np.zeros(case["phases"])
    st["out"] = [_tensor(f["dst"]) for f in st["cent"] + st["vert"]] + [_tensor(p) for p in st["perc"]]
    return st


def _run_markers(st):
    c = st["ctx"]
    c.markers_set(st["x"], st["z"], st["ph"])
    c.p2mastah_fused(1, st["stencil"], st["cent"])
    c.p2mastah_fused(0, st["stencil"], st["vert"])
    c.p2mastah(st["none"], prop=1, centroid=1, interp_stencil=st["stencil"], nb_phases=st["nph"],
               phase_perc=st["perc"])
    return st["out"]


def _exact_markers(case, seed):
    x, z, ph, T = _markers_inputs(case, seed)
    g = _coords(case)
    nx, nz = case["nx"], case["nz"]
    eta, rho, G = (torch.as_tensor(t, device="cuda")[ph.long()] for t in _tables(case))
    R = 1 if case["stencil"] == 9 else 0
    hx, hz = g["dx"] * (1.5 if R else 0.5), g["dz"] * (1.5 if R else 0.5)

    def sums(X, Z, mx, mz, fields):
        i0 = (torch.ceil((x - X[0]) / g["dx"] + 0.5).long() - 1).clamp(0, mx - 1)
        j0 = (torch.ceil((z - Z[0]) / g["dz"] + 0.5).long() - 1).clamp(0, mz - 1)
        acc = [torch.zeros(mx * mz, dtype=F64, device="cuda") for _ in range(len(fields) + 1)]
        for dj in range(-R, R + 1):
            for di in range(-R, R + 1):
                i, j = i0 + di, j0 + dj
                ok = (i >= 0) & (i < mx) & (j >= 0) & (j < mz)
                w = (1.0 - (X[i0] + di * g["dx"] - x).abs() / hx) * (1.0 - (Z[j0] + dj * g["dz"] - z).abs() / hz)
                w = torch.where(ok, w, torch.zeros_like(w))
                at = i.clamp(0, mx - 1) + j.clamp(0, mz - 1) * mx
                acc[0].index_add_(0, at, w)
                for a, f in zip(acc[1:], fields):
                    a.index_add_(0, at, w * f)
        W = acc[0]
        return [torch.where(W.abs() < 1e-30, torch.zeros_like(W), a / W) for a in acc[1:]]

    def back(v, avg):
        if avg == 0:
            return v
        return torch.where(v == 0, v, 1.0 / v) if avg == 1 else torch.where(v == 0, v, torch.exp(v))

    fc = [torch.log(eta), rho, 1.0 / G, T] + [(ph == p).double() for p in range(case["phases"])]
    c = sums(g["xc"], g["zc"], nx, nz, fc)
    v = sums(g["xg"], g["zg"], nx + 1, nz + 1, fc[:3])
    return ([back(c[0], 2), c[1], back(c[2], 1), c[3], back(v[0], 2), v[1], back(v[2], 1)] + c[4:])


# ------------------------------------------------------------------- advect
def _advect_inputs(case, seed):
    gen = _gen(seed)
    x, z = _positions(case, gen, False)
    g = _coords(case)
    Lx, Lz = _box(case)[1], _box(case)[3]
    u = (torch.sin(math.pi * g["xg"] / Lx)[None, :] * torch.cos(math.pi * g["zvx"] / Lz)[:, None])
    v = -(Lz / Lx) * (torch.cos(math.pi * g["xvz"] / Lx)[None, :] * torch.sin(math.pi * g["zg"] / Lz)[:, None])
    nc, nv = case["nx"] * case["nz"], (case["nx"] + 1) * (case["nz"] + 1)
    grids = [_uniform(gen, m, -1.0, 1.0) for m in (nc, nc, nc, nc, nv, nc, nc, nv)]   # p, p0, sxx.., sxx0..
    mark = [_uniform(gen, x.numel(), -1.0, 1.0) for _ in range(4)]                     # P, sxx, szz, sxz
    return x, z, u.reshape(-1), v.reshape(-1), grids, mark, 0.5 * g["dx"]


def _prepare_advect(case, seed):
    x, z, u, v, grids, mark, dt = _advect_inputs(case, seed)
    c = _context(case)
    n = x.numel()
    st = dict(ctx=c, x=_upload(c, x), z=_upload(c, z), ph=_upload(c, torch.zeros(n, dtype=torch.int32, device="cuda")),
              u=_upload(c, u), v=_upload(c, v), vx=_zeros(c, n), vz=_zeros(c, n), dt=dt, conserv=case["conserv"],
              grids=[_upload(c, a) for a in grids], mark=[_upload(c, a) for a in mark])
    st["out"] = [_tensor(st[k]) for k in ("x", "z", "ph", "vx", "vz")] + [_tensor(a) for a in st["mark"]]
    return st


def _run_advect(st):
    c, G, m = st["ctx"], st["grids"], st["mark"]
    x, z, ph = st["x"], st["z"], st["ph"]
    c.update_particle_pressure(G[0], G[1], x, z, ph, m[0])
    c.update_particle_stress(G[2], G[3], G[4], G[5], G[6], G[7], x, z, ph, m[1], m[2], m[3])
    c.advect_rk4(st["u"], st["v"], st["dt"], x, z, ph, st["conserv"], st["vx"], st["vz"])
    st["dt"] = -st["dt"]     # to and fro, so that any number of passes leaves the markers as they were laid out
    return st["out"]


def _exact_advect(case, seed):
    x, z, u, v, G, mark, dt = _advect_inputs(case, seed)
    g = _coords(case)
    dx, dz = g["dx"], g["dz"]

    def cell(p, X, h, n, lo, hi):
        j = (torch.ceil((p - X[0]) / h).long() - 1).clamp(lo, hi)
        return j

    def along(F, n, at, step, t, j, last, conserv):
        """Interpolation along one axis, with the correction of the second difference."""
        a, b = F[at], F[at + step]
        r = a * (1.0 - t) + b * t
        if conserv:
            up, dn = (t >= 0.5) & (j < last), (t < 0.5) & (j > 0)
            far = F[torch.where(up, at + 2 * step, torch.where(dn, at - step, at))]
            d2 = torch.where(up, a - 2.0 * b + far, torch.where(dn, far - 2.0 * a + b, torch.zeros_like(a)))
            r = r + 0.5 * (t - 0.5) ** 2 * d2
        return r

    def vel(p, q):
        Nx, Nz = case["nx"] + 1, case["nz"] + 2
        j, i = cell(p, g["xg"], dx, Nx, 0, Nx - 2), cell(q, g["zvx"], dz, Nz, 0, Nz - 2)
        t, s, at = (p - g["xg"][j]).abs() / dx, (q - g["zvx"][i]).abs() / dz, j + i * Nx
        a = (1.0 - s) * along(u, Nx, at, 1, t, j, Nx - 2, case["conserv"]) + \
            s * along(u, Nx, at + Nx, 1, t, j, Nx - 2, case["conserv"])
        Nx, Nz = case["nx"] + 2, case["nz"] + 1
        j, i = cell(p, g["xvz"], dx, Nx, 0, Nx - 2), cell(q, g["zg"], dz, Nz, 0, Nz - 2)
        t, s, at = (p - g["xvz"][j]).abs() / dx, (q - g["zg"][i]).abs() / dz, j + i * Nx
        b = (1.0 - t) * along(v, Nx, at, Nx, s, i, Nz - 2, case["conserv"]) + \
            t * along(v, Nx, at + 1, Nx, s, i, Nz - 2, case["conserv"])
        return a, b

    def centres(F):
        n, m = case["nx"], case["nz"]
        P = torch.nn.functional.pad(F.reshape(1, 1, m, n), (1, 1, 1, 1), mode="replicate").reshape(-1)
        j, i = cell(x, g["xvz"], dx, n, 0, n), cell(z, g["zvx"], dz, m, 0, m)
        t, s, at, w = (x - g["xvz"][j]) / dx, (z - g["zvx"][i]) / dz, j + i * (n + 2), n + 2
        return (1 - t) * (1 - s) * P[at] + t * (1 - s) * P[at + 1] + (1 - t) * s * P[at + w] + t * s * P[at + w + 1]

    def vertices(F):
        n, m = case["nx"] + 1, case["nz"] + 1
        j, i = cell(x, g["xg"], dx, n, 0, n - 2), cell(z, g["zg"], dz, m, 0, m - 2)
        t, s, at = (x - g["xg"][j]).abs() / dx, (z - g["zg"][i]).abs() / dz, j + i * n
        return (1 - t) * (1 - s) * F[at] + t * (1 - s) * F[at + 1] + (1 - t) * s * F[at + n] + t * s * F[at + n + 1]

    m = [mark[0] + centres(G[0] - G[1]), mark[1] + centres(G[2] - G[5]), mark[2] + centres(G[3] - G[6]),
         mark[3] + vertices(G[4] - G[7])]
    a1, b1 = vel(x, z)
    a2, b2 = vel(x + 0.5 * dt * a1, z + 0.5 * dt * b1)
    a3, b3 = vel(x + 0.5 * dt * a2, z + 0.5 * dt * b2)
    a4, b4 = vel(x + dt * a3, z + dt * b3)
    vx, vz = (a1 + 2 * a2 + 2 * a3 + a4) / 6, (b1 + 2 * b2 + 2 * b3 + b4) / 6
    return [x + dt * vx, z + dt * vz, None, vx, vz] + m


# ----------------------------------------------------------------- rheology
def _laws(law):
    """Phase tables in scaled units, and the call's parameters."""
    zero = {k: 0.0 for k in mdgpu.LAW_TAIL}
    if law == "vep":
        ph = [dict(zero, **d) for d in S.vep_phases(C=1.0)]
        prm = dict(average=0, step=1, elastic=1, dt=1.0, R=1.0, zeroC=0.0, min_eta=1e-4, max_eta=1e4, eta_tol=1e-13,
                   Tiimin=1e-5, scale_E=1.0, scale_eta=1.0)
    else:
        base = dict(zero, cstv=0, pwlv=1, plast=1, eta0=1.0, pref_pwl=1.0, F_pwl=1.0, A_pwl=1.0, n_pwl=3.0, Q_pwl=3.0,
                    V_pwl=0.05, C=3.0, fric=math.radians(30.0), dil=0.0, Slim=20.0, eta_vp=0.0, n_vp=1.0, beta=1e-50,
                    f_pwl=1.0, f_lin=1.0, f_gbs=1.0, gs_ref=1.0)
        mantle = dict(base, n_pwl=3.5, Q_pwl=5.0, linv=1, F_lin=1.0, A_lin=2.0, n_lin=1.0, m_lin=3.0, Q_lin=4.0,
                      V_lin=0.03, expv=1, G_exp=0.1, S_exp=60.0, Q_exp=12.0, E_exp=1e3, n_exp=2.0, a_pwl=20.0, a_lin=30.0)
        ph = [base, dict(base, A_pwl=0.5, Q_pwl=4.0, C=4.0), mantle]
        prm = dict(average=1, step=1, elastic=1, dt=2.0, R=1.0, zeroC=0.2, min_eta=1e-4, max_eta=1e4, eta_tol=1e-13,
                   Tiimin=1e-5, scale_E=1.0, scale_eta=1.0, T_peierls=1.0, d_min=1e-9)
    return ph, prm


def _rheology_inputs(case, seed):
    """Layers (or weak seeds) whose boundaries cross cells, a smooth flow
    with a jitter, old stresses near yield."""
    gen = _gen(seed)
    g = _coords(case)
    law = case["law"]
    nph = 2 if law == "vep" else 3
    Lx, Lz = _box(case)[1], _box(case)[3]
    r = torch.rand(64, 2, dtype=F64, device="cuda", generator=gen)

    def fractions(X, Z):
        xx, zz = X[None, :].expand(len(Z), len(X)), Z[:, None].expand(len(Z), len(X))
        if law == "vep":
            d = torch.full_like(xx, 1e9)
            for k in range(64):
                d = torch.minimum(d, torch.sqrt((xx - Lx * r[k, 0]) ** 2 + (zz - Lz * r[k, 1]) ** 2))
            w = ((2.5 * g["dx"] - d) / g["dx"]).clamp(0.0, 1.0)
            return torch.stack([1.0 - w, w]).reshape(2, -1)
        h = zz + 0.02 * torch.sin(9.0 * xx)
        a = ((h - 0.65 * Lz) / g["dz"] + 0.5).clamp(0.0, 1.0)     # upper crust
        b = ((0.35 * Lz - h) / g["dz"] + 0.5).clamp(0.0, 1.0)     # mantle
        return torch.stack([a, 1.0 - a - b, b]).reshape(3, -1)

    d = dict(perc_n=fractions(g["xc"], g["zc"]), perc_s=fractions(g["xg"], g["zg"]))
    nc, nv = case["nx"] * case["nz"], (case["nx"] + 1) * (case["nz"] + 1)

    def noise(m, s):
        return torch.randn(m, dtype=F64, device="cuda", generator=gen) * s

    u = -g["xg"][None, :].expand(case["nz"] + 2, -1).reshape(-1)
    v = g["zg"][:, None].expand(-1, case["nx"] + 2).reshape(-1)
    d["u"] = u + noise(u.numel(), 0.2 * g["dx"])
    d["v"] = v + noise(v.numel(), 0.2 * g["dz"])
    zc = g["zc"][:, None].expand(-1, case["nx"]).reshape(-1) / Lz
    d["T"] = (1.6 - 1.1 * zc) + noise(nc, 0.02) if law == "creep" else torch.ones(nc, dtype=F64, device="cuda")
    d["p"] = (6.0 * (1.0 - zc) if law == "creep" else 0.5 + 0.0 * zc) + noise(nc, 0.1)
    for s, m in (("n", nc), ("s", nv)):
        d["G_" + s] = torch.ones(m, dtype=F64, device="cuda")
        d["xx0_" + s] = 0.2 + noise(m, 0.05)
        d["zz0_" + s] = -d["xx0_" + s]
        d["xz0_" + s] = noise(m, 0.02)
        if law == "vep":
            d["pref_" + s] = torch.exp(noise(m, 0.5))
        else:
            d["d_" + s] = torch.exp(noise(m, 0.3))
            d["phi_" + s] = (torch.rand(m, dtype=F64, device="cuda", generator=gen) - 0.9).clamp(min=0.0) * 0.2
    d["rx"] = noise(u.numel(), 1.0)
    d["rz"] = noise(v.numel(), 1.0)
    return d


def _prepare_rheology(case, seed):
    d = _rheology_inputs(case, seed)
    c = _context(case)
    A = {k: _upload(c, t) for k, t in d.items()}
    ph, prm = _laws(case["law"])
    nc, nv, neq = c.node_count(1), c.node_count(0), c.eqn_count()[0]
    st = dict(ctx=c, A=A, phases=[mdgpu.PhaseProp(**p) for p in ph], prm=mdgpu.RheoParams(**prm), newton=case["newton"],
              sr={k: _zeros(c, nv if k == "exz" else nc) for k in ("div", "exxd", "ezzd", "exz")},
              nodes={k: _zeros(c, nc if k == "exz_n" else nv) for k in ("exz_n", "exxd_s", "ezzd_s", "div_s")},
              cen={k: _zeros(c, nc) for k in mdgpu.RHEO_OUT}, ver={k: _zeros(c, nv) for k in mdgpu.RHEO_OUT},
              T_s=_zeros(c, nv), P_s=_zeros(c, nv), F=_zeros(c, neq))
    if case["newton"]:
        st["Dn"], st["Ds"] = _zeros(c, 8 * nc), _zeros(c, 4 * nv)
    st["view"] = dict(F=_tensor(st["F"]))
    for s in ("cen", "ver"):
        for k in ("eta", "eta_phys", "sxx", "szz", "sxz", "p_corr", "eII_pl"):
            st["view"][s + "_" + k] = _tensor(st[s][k])
    if case["newton"]:
        st["view"]["Dn"], st["view"]["Ds"] = _tensor(st["Dn"]), _tensor(st["Ds"])
    return st


def _run_rheology(st):
    c, A, sr, nd = st["ctx"], st["A"], st["sr"], st["nodes"]
    c.apply_bc(A["u"], A["v"])
    c.strain_rates(A["u"], A["v"], out=sr)
    c.strain_rates_nodes(sr["exxd"], sr["ezzd"], sr["exz"], sr["div"], out=nd)
    c.c2v(A["T"], st["T_s"])
    c.c2v(A["p"], st["P_s"])
    node = {}
    for s, k in (("n", 1), ("s", 0)):
        e = (sr["exxd"], sr["ezzd"], nd["exz_n"]) if k else (nd["exxd_s"], nd["ezzd_s"], sr["exz"])
        a = dict(perc=A["perc_" + s], G=A["G_" + s], T=A["T"] if k else st["T_s"], P=A["p"] if k else st["P_s"],
                 exx=e[0], ezz=e[1], exz=e[2], sxx0=A["xx0_" + s], szz0=A["zz0_" + s], sxz0=A["xz0_" + s])
        for f in ("pref", "d", "phi"):
            if f + "_" + s in A:
                a[f] = A[f + "_" + s]
        node[k] = a
        c.viscosity_grid(st["phases"], st["prm"], k, **a, **(st["cen"] if k else st["ver"]))
    _, norms = c.stokes_residual(st["cen"]["sxx"], st["cen"]["szz"], st["ver"]["sxz"], st["cen"]["p_corr"], sr["div"],
                                 A["rx"], A["rz"], F=st["F"])
    if st["newton"]:
        c.tangent_grid(st["phases"], st["prm"], 1, D=st["Dn"], **node[1])
        c.tangent_grid(st["phases"], st["prm"], 0, D=st["Ds"], **node[0])
    return dict(st["view"], norms=norms)


def _viscosity(m, prm, G, T, P, d, phi, pref, Exx, Ezz, Exz):
    """One phase's effective and dissipative viscosity, plastic strain rate
    (no dilation, no viscoplastic regularisation)."""
    Eii = torch.sqrt(0.5 * (Exx ** 2 + Ezz ** 2 + (Exx + Ezz) ** 2) + Exz ** 2).clamp(min=1e-30)
    T0, T = T, T.clamp(min=prm["zeroC"])
    eel = G * prm["dt"]
    n = m["n_pwl"]
    B = m["pref_pwl"] * pref * m["F_pwl"] * m["A_pwl"] ** (-1.0 / n) * torch.exp((m["Q_pwl"] + P * m["V_pwl"]) / (n * T)) * \
        d ** (m["m_pwl"] / n) * torch.exp(-m["a_pwl"] * phi / n)
    terms = [((2.0 * B) ** -n, torch.full_like(T, n), B)]
    if m.get("linv"):
        nl = m["n_lin"]
        Bl = m["F_lin"] * m["A_lin"] ** (-1.0 / nl) * torch.exp((m["Q_lin"] + P * m["V_lin"]) / (nl * T)) * \
            torch.exp(-m["a_lin"] * phi / nl)
        terms.append(((2.0 * Bl) ** -nl * d ** -m["m_lin"], torch.full_like(T, nl),
                      Bl * m["gs_ref"] ** (m["m_lin"] / nl)))
    if m.get("expv"):
        g = m["G_exp"]
        ST = m["Q_exp"] / T * 2.0 * g * (1.0 - g)
        q = ST + m["n_exp"]
        arr = torch.exp(-m["Q_exp"] / T * (1.0 - g) ** 2)
        F = (2.0 ** (1.0 - q) / math.sqrt(3.0) ** (q + 1.0)) ** (1.0 / q)
        Be = F * (g * m["S_exp"]) ** (ST / q) / (m["E_exp"] * arr) ** (1.0 / q)
        on = T0 < prm["T_peierls"]
        terms.append((torch.where(on, (2.0 * Be) ** -q, torch.zeros_like(q)), q,
                      torch.where(on, Be, torch.full_like(Be, math.inf))))
    # the stress that the rates add up to the given one: Newton on its logarithm
    tau = 2.0 * eel * Eii
    for C, q, _ in terms:
        tau = torch.minimum(tau, torch.where(C > 0, (Eii / C.clamp(min=1e-300)) ** (1.0 / q), tau))
    for _ in range(60):
        f, df = tau / (2.0 * eel), tau / (2.0 * eel)
        for C, q, _B in terms:
            e = C * tau ** q
            f, df = f + e, df + q * e
        tau = tau * torch.exp((torch.log(Eii) - torch.log(f)) * f / df)
    eta_ve = tau / (2.0 * Eii)
    inv = torch.zeros_like(tau)
    for C, q, Bq in terms:
        inv = inv + torch.where(C > 0, 1.0 / (Bq * (C * tau ** q).clamp(min=1e-300) ** (1.0 / q - 1.0)),
                                torch.zeros_like(tau))
    Ty = (m["C"] * math.cos(m["fric"]) + P * math.sin(m["fric"])).clamp(max=m["Slim"])
    pl = (tau - Ty) > 1e-17
    Tn = torch.where(Ty < 0, torch.full_like(Ty, prm["Tiimin"]), Ty)
    gdot = torch.where(pl, (tau - Tn) / eta_ve, torch.zeros_like(tau))
    eta = torch.where(pl, Tn / (2.0 * Eii), eta_ve)
    inv = inv + torch.where(pl, gdot / Tn, torch.zeros_like(tau))
    return eta.clamp(prm["min_eta"], prm["max_eta"]), (1.0 / inv).clamp(prm["min_eta"], prm["max_eta"]), gdot / 2.0


def _exact_rheology(case, seed):
    d = _rheology_inputs(case, seed)
    g = _coords(case)
    dx, dz, nx, nz = g["dx"], g["dz"], case["nx"], case["nz"]
    u, v = d["u"].reshape(nz + 2, nx + 1).clone(), d["v"].reshape(nz + 1, nx + 2).clone()
    u[0], u[-1], v[:, 0], v[:, -1] = u[1], u[-2], v[:, 1], v[:, -2]
    exx, ezz = (u[1:-1, 1:] - u[1:-1, :-1]) / dx, (v[1:, 1:-1] - v[:-1, 1:-1]) / dz
    exz = 0.5 * ((u[1:] - u[:-1]) / dz + (v[:, 1:] - v[:, :-1]) / dx)
    div = exx + ezz

    def c2v(a):
        a = torch.nn.functional.pad(a.reshape(1, 1, nz, nx), (1, 1, 1, 1), mode="replicate")[0, 0]
        return 0.25 * (a[1:, 1:] + a[1:, :-1] + a[:-1, 1:] + a[:-1, :-1])

    exz_n = 0.25 * (exz[1:, 1:] + exz[1:, :-1] + exz[:-1, 1:] + exz[:-1, :-1])
    ph, prm = _laws(case["law"])
    out = {}
    for s, name, E in (("n", "cen", (exx, ezz, exz_n)), ("s", "ver", (c2v(exx), c2v(ezz), exz))):
        T, P = (d["T"], d["p"]) if s == "n" else (c2v(d["T"]).reshape(-1), c2v(d["p"]).reshape(-1))
        G, ee = d["G_" + s], prm["dt"] * d["G_" + s]
        X, Z, XZ = (e.reshape(-1) + d[k + "0_" + s] / ee / 2.0 for e, k in zip(E, ("xx", "zz", "xz")))
        one = torch.ones_like(T)
        pref, gs, phi = d.get("pref_" + s, one), d.get("d_" + s, one), d.get("phi_" + s, 0.0 * one)
        e, ep, epl = 0.0 * one, 0.0 * one, 0.0 * one
        for i, m in enumerate(ph):
            w = d["perc_" + s][i]
            w = torch.where(w.abs() > 1e-13, w, torch.zeros_like(w))
            a, b, c = _viscosity(m, prm, G, T, P, gs, phi, pref, X, Z, XZ)
            e, ep = (e + w * a, ep + w * b) if prm["average"] == 0 else (e + w / a, ep + w / b)
            epl = epl + w * c
        if prm["average"] == 1:
            e, ep = 1.0 / e, 1.0 / ep
        tot = sum(torch.where(w.abs() > 1e-13, w, torch.zeros_like(w)) for w in d["perc_" + s])
        out.update({name + "_" + k: t for k, t in dict(eta=e, eta_phys=ep, sxx=2 * e * X, szz=2 * e * Z, sxz=2 * e * XZ,
                                                        p_corr=tot * P, eII_pl=epl).items()})
    # residual in equation numbering
    sxx, szz, pc = (out["cen_" + k].reshape(nz, nx) for k in ("sxx", "szz", "p_corr"))
    sxz = out["ver_sxz"].reshape(nz + 1, nx + 1)
    rx, rz = d["rx"].reshape(nz + 2, nx + 1), d["rz"].reshape(nz + 1, nx + 2)
    s1, s2 = sxx - pc, szz - pc
    fx = (s1[:, 1:] - s1[:, :-1]) / dx + (sxz[1:, 1:-1] - sxz[:-1, 1:-1]) / dz + rx[1:-1, 1:-1]
    fz = (s2[1:] - s2[:-1]) / dz + (sxz[1:-1, 1:] - sxz[1:-1, :-1]) / dx + rz[1:-1, 1:-1]
    V = dx * dz
    out["F"] = torch.cat([-V * fx.reshape(-1), -V * fz.reshape(-1), V * div.reshape(-1)])
    a, b = V * fx[2:-1], V * fz[:, 2:-1]    # rows and columns nearest the walls do not enter the norms
    out["norms"] = torch.stack([a.square().mean().sqrt(), b.square().mean().sqrt(), (V * div).square().mean().sqrt()])
    if case["newton"]:
        out["Dn"], out["Ds"] = None, None   # finite differences of the viscosity, no 64-bit value of their own
    return out


# -------------------------------------------------------------------- solve
def _solve_inputs(case, seed):
    """Nodal viscosities (geometric means over 3 x 3 points of a cell) and
    densities of seeded ellipses with a contrast of 1e6, or of one inclusion
    of viscosity 1e3."""
    gen = _gen(seed)
    g = _coords(case)
    Lx, Lz = _box(case)[1], _box(case)[3]
    h = g["dx"]
    m = 256 if case["body"] == "ellipses" else 1
    m = max(4, int(round(m * case["nx"] * case["nz"] / 2047.0 ** 2))) if m > 1 else 1
    p = torch.rand((m, 7), dtype=F64, device="cuda", generator=gen).cpu().numpy()

    def at(x, z):
        le, rho = torch.zeros_like(x), torch.full_like(x, 3000.0)
        for i in range(m):
            if case["body"] == "ellipses":
                cx, cz, th = Lx * p[i, 0], Lz * p[i, 1], math.pi * p[i, 4]
                a, b = 0.5 * h * (5 + 55 * p[i, 2]), 0.5 * h * (5 + 55 * p[i, 3])
                val, den = math.log(10.0) * (6 * p[i, 5] - 3), 2700.0 + 600.0 * p[i, 6]
            else:
                cx, cz, th = Lx * (0.45 + 0.1 * p[i, 0]), Lz * (0.45 + 0.1 * p[i, 1]), math.pi * p[i, 4]
                a, b = 0.2 + 0.02 * p[i, 2], 0.2 + 0.02 * p[i, 3]
                val, den = math.log(1e3), 3000.0
            c, s = math.cos(th), math.sin(th)
            inside = ((c * (x - cx) + s * (z - cz)) / a) ** 2 + ((c * (z - cz) - s * (x - cx)) / b) ** 2 <= 1.0
            le, rho = torch.where(inside, torch.full_like(le, val), le), torch.where(inside, torch.full_like(le, den), rho)
        return le, rho

    def nodes(X, Z):
        le, rho = 0.0, 0.0
        for a in (-1, 0, 1):
            for b in (-1, 0, 1):
                e, r = at((X[None, :] + a * h / 3).expand(len(Z), -1), (Z[:, None] + b * g["dz"] / 3).expand(-1, len(X)))
                le, rho = le + e / 9.0, rho + r / 9.0
        return torch.exp(le), rho

    en, rn = nodes(g["xc"], g["zc"])
    es, _ = nodes(g["xg"], g["zg"])
    dx, dz = g["dx"], g["dz"]
    V = dx * dz
    nx, nz = case["nx"], case["nz"]
    if case["body"] == "ellipses":      # body force at rest
        fx = torch.zeros((nz, nx - 1), dtype=F64, device="cuda")
        fz = -9.81 * 0.5 * (rn[1:] + rn[:-1])
    else:                               # pure shear: exx = -1, ezz = 1
        fx, fz = (-2.0 * en[:, 1:] + 2.0 * en[:, :-1]) / dx, (2.0 * en[1:] - 2.0 * en[:-1]) / dz
    F = torch.cat([-V * fx.reshape(-1), -V * fz.reshape(-1), torch.zeros(nx * nz, dtype=F64, device="cuda")])
    return en, es, F


def _prepare_solve(case, seed):
    en, es, F = _solve_inputs(case, seed)
    c = _context(case)
    opts = {"default": {}, "patch": PATCH, "patch_mixed": PATCH_MIXED}[case["opts"]]
    st = dict(ctx=c, D11=_upload(c, 2.0 * en), D33=_upload(c, es), F=_upload(c, F), sol=_zeros(c, F.numel()),
              nm=c.eqn_count()[1], opts=opts)
    st["out"] = _tensor(st["sol"])
    return st


def _run_solve(st):
    st["ctx"].killer_solver_dev(st["D11"], st["D11"], st["D33"], st["F"], st["nm"], st["sol"], **st["opts"])
    return st["out"]


def _exact_solve(case, seed):
    """Block elimination of the Picard system row by row (each row of cells
    with its Vx and its upper Vz), then refinement with the residual."""
    nx, nz = case["nx"], case["nz"]
    if nx > 160 or nz > 400:
        return None
    en, es, F = (t.cpu().numpy() for t in _solve_inputs(case, seed))
    g = _coords(case)
    dx, dz = g["dx"], g["dz"]
    V = dx * dz
    nu, nv = nz * (nx - 1), (nz - 1) * nx
    n = nu + nv + nx * nz
    iu = np.full((nz + 2, nx + 1), -1)
    iu[1:-1, 1:-1] = np.arange(nu).reshape(nz, nx - 1)
    iv = np.full((nz + 1, nx + 2), -1)
    iv[1:-1, 1:-1] = nu + np.arange(nv).reshape(nz - 1, nx)
    ip = nu + nv + np.arange(nx * nz).reshape(nz, nx)
    R, Cc, A = [], [], []

    def put(r, c, a):
        r, c, a = np.broadcast_arrays(r, c, a)
        ok = c >= 0
        R.append(r[ok]), Cc.append(c[ok]), A.append(a[ok])

    r = iu[1:-1, 1:-1]
    W, E, Sv, Nv = 2 * en[:, :-1] / dx ** 2, 2 * en[:, 1:] / dx ** 2, es[:-1, 1:-1].copy(), es[1:, 1:-1].copy()
    cS, cN = Sv / (dx * dz), Nv / (dx * dz)
    Sv, Nv = Sv / dz ** 2, Nv / dz ** 2
    Sv[0], Nv[-1] = 0.0, 0.0             # free slip
    put(r, r, V * (W + E + Sv + Nv))
    put(r, iu[1:-1, :-2], -V * W), put(r, iu[1:-1, 2:], -V * E), put(r, iu[:-2, 1:-1], -V * Sv)
    put(r, iu[2:, 1:-1], -V * Nv)
    put(r, iv[:-1, 1:-2], -V * cS), put(r, iv[:-1, 2:-1], V * cS), put(r, iv[1:, 1:-2], V * cN)
    put(r, iv[1:, 2:-1], -V * cN)
    put(r, ip[:, :-1], -V / dx), put(r, ip[:, 1:], V / dx)
    r = iv[1:-1, 1:-1]
    Sc, Nc, W, E = 2 * en[:-1] / dz ** 2, 2 * en[1:] / dz ** 2, es[1:-1, :-1].copy(), es[1:-1, 1:].copy()
    cW, cE = W / (dx * dz), E / (dx * dz)
    W, E = W / dx ** 2, E / dx ** 2
    W[:, 0], E[:, -1] = 0.0, 0.0
    put(r, r, V * (Sc + Nc + W + E))
    put(r, iv[:-2, 1:-1], -V * Sc), put(r, iv[2:, 1:-1], -V * Nc), put(r, iv[1:-1, :-2], -V * W)
    put(r, iv[1:-1, 2:], -V * E)
    put(r, iu[1:-2, :-1], -V * cW), put(r, iu[1:-2, 1:], V * cE), put(r, iu[2:-1, :-1], V * cW)
    put(r, iu[2:-1, 1:], -V * cE)
    put(r, ip[:-1], -V / dz), put(r, ip[1:], V / dz)
    put(ip, iu[1:-1, :-1], -V / dx), put(ip, iu[1:-1, 1:], V / dx)
    put(ip, iv[:-1, 1:-1], -V / dz), put(ip, iv[1:, 1:-1], V / dz)
    R, Cc, A = (np.concatenate([a.ravel() for a in q]) for q in (R, Cc, A))
    pin = ip[-1, -1]                     # the free constant of the pressure
    keep = R != pin
    R, Cc, A = np.append(R[keep], pin), np.append(Cc[keep], pin), np.append(A[keep], 1.0)
    rhs = F.copy()
    rhs[pin] = 0.0
    row = np.empty(n, int)
    row[iu[1:-1, 1:-1]] = np.arange(nz)[:, None]
    row[iv[1:-1, 1:-1]] = np.arange(nz - 1)[:, None]
    row[ip] = np.arange(nz)[:, None]
    order = np.argsort(row, kind="stable")
    count = np.bincount(row, minlength=nz)
    first = np.concatenate([[0], np.cumsum(count)])
    loc = np.empty(n, int)
    loc[order] = np.arange(n) - first[row[order]]
    mats = {}
    for dlt in (-1, 0, 1):
        m = row[Cc] - row[R] == dlt
        byrow = np.argsort(row[R[m]], kind="stable")
        mats[dlt] = (R[m][byrow], Cc[m][byrow], A[m][byrow],
                     np.concatenate([[0], np.cumsum(np.bincount(row[R[m]], minlength=nz))]))

    def block(dlt, l):
        r, c, a, off = mats[dlt]
        s = slice(off[l], off[l + 1])
        M = np.zeros((count[l], count[l + dlt]))
        np.add.at(M, (loc[r[s]], loc[c[s]]), a[s])
        return M

    inv, up, low = [], [], []
    for l in range(nz):
        D = block(0, l)
        lo = block(-1, l) if l else None
        if l:
            D = D - lo @ up[-1]
        low.append(lo)
        inv.append(np.linalg.inv(D))
        up.append(inv[-1] @ block(1, l) if l + 1 < nz else None)

    def solve(b):
        y, x = [], np.empty(n)
        for l in range(nz):
            t = b[order[first[l]:first[l + 1]]]
            y.append(inv[l] @ (t - low[l] @ y[-1] if l else t))
        for l in reversed(range(nz)):
            z = y[l] - (up[l] @ z if l + 1 < nz else 0.0)
            x[order[first[l]:first[l + 1]]] = z
        return x

    x = np.zeros(n)
    for _ in range(5):
        res = rhs - np.bincount(R, weights=A * x[Cc], minlength=n)
        x = x + solve(res)
    res = rhs - np.bincount(R, weights=A * x[Cc], minlength=n)
    if not np.linalg.norm(res) < 1e-9 * np.linalg.norm(rhs):
        return None
    x[nu + nv:] -= x[nu + nv:].mean()
    return torch.as_tensor(x)


# ------------------------------------------------------------------- energy
def _energy_inputs(case, seed):
    gen = _gen(seed)
    nx, nz = case["nx"], case["nz"]
    nc = nx * nz
    h = 1.0 / max(nx, nz)
    d = dict(rho=_uniform(gen, nc, 2.5, 3.5), Cp=_uniform(gen, nc, 900.0, 1100.0),
             kx=_uniform(gen, (nx + 1) * (nz + 2), 1.0, 5.0), kz=_uniform(gen, (nx + 2) * (nz + 1), 1.0, 5.0),
             Qr=_uniform(gen, nc, 0.0, 1e3), Wdiss=_uniform(gen, nc, 0.0, 1e3))
    zc = (torch.arange(nz, dtype=F64, device="cuda") + 0.5) / nz
    d["T"] = (1603.0 - 1330.0 * zc)[:, None].expand(nz, nx).reshape(-1) + _uniform(gen, nc, -20.0, 20.0)
    BT = torch.zeros((nz + 2, nx + 2), dtype=torch.int8, device="cuda")
    BV = torch.zeros((nz + 2, nx + 2), dtype=F64, device="cuda")
    BT[-1], BV[-1] = 1, 273.0           # surface and base held, insulated sides
    BT[0], BV[0] = 1, 1603.0
    d["BT"], d["BV"] = BT.reshape(-1), BV.reshape(-1)
    return d, case["fourier"] * h * h * 3.0 * 1000.0 / 3.0


def _prepare_energy(case, seed):
    d, dt = _energy_inputs(case, seed)
    c = _context(case)
    st = dict(ctx=c, dt=dt, A={k: _upload(c, t) for k, t in d.items()}, T=_zeros(c, d["T"].numel()))
    st["out"] = _tensor(st["T"])
    return st


def _run_energy(st):
    A = st["A"]
    st["T"].copy_from(A["T"])           # the old temperature is kept beside the new one
    st["ctx"].energy_step(st["dt"], A["rho"], A["Cp"], st["T"], A["kx"], A["kz"], A["BT"], A["BV"], Qr=A["Qr"],
                          Wdiss=A["Wdiss"])
    return st["out"]


def _exact_energy(case, seed):
    d, dt = _energy_inputs(case, seed)
    nx, nz = case["nx"], case["nz"]
    x0, x1, z0, z1 = _box(case)
    dx, dz = (x1 - x0) / nx, (z1 - z0) / nz
    kx, kz = d["kx"].reshape(nz + 2, nx + 1)[1:-1].clone() / dx ** 2, d["kz"].reshape(nz + 1, nx + 2)[:, 1:-1] / dz ** 2
    kx[:, 0], kx[:, -1] = 0.0, 0.0
    BV = d["BV"].reshape(nz + 2, nx + 2)
    m = (d["rho"] * d["Cp"]).reshape(nz, nx) / dt
    b = m * d["T"].reshape(nz, nx) + (d["Qr"] + d["Wdiss"]).reshape(nz, nx)
    b[0] += 2.0 * kz[0] * BV[0, 1:-1]
    b[-1] += 2.0 * kz[-1] * BV[-1, 1:-1]
    diag = m + kx[:, 1:] + kx[:, :-1] + kz[1:] + kz[:-1]
    diag[0] += kz[0]
    diag[-1] += kz[-1]

    def mul(x):
        y = diag * x
        y[:, 1:] -= kx[:, 1:-1] * x[:, :-1]
        y[:, :-1] -= kx[:, 1:-1] * x[:, 1:]
        y[1:] -= kz[1:-1] * x[:-1]
        y[:-1] -= kz[1:-1] * x[1:]
        return y

    x = d["T"].reshape(nz, nx).clone()
    for _ in range(2):                  # restarted once from the true residual
        r = b - mul(x)
        z = r / diag
        p, rz = z.clone(), (r * z).sum()
        end = 1e-30 * (b * b / diag).sum()
        for it in range(3000):
            q = mul(p)
            a = rz / (p * q).sum()
            x = x + a * p
            r = r - a * q
            z = r / diag
            new = (r * z).sum()
            if it % 16 == 0 and new < end:
                break
            p, rz = z + (new / rz) * p, new
    return x.reshape(-1)


# ------------------------------------------------------------------ network
def _network_inputs(case, seed):
    gen = _gen(seed)
    n = case["h"] * case["w"] * 4
    x, t = (torch.randn(n, dtype=torch.float32, device="cuda", generator=gen) for _ in range(2))
    mask = torch.ones((case["h"], case["w"], 4), dtype=torch.float32, device="cuda")
    mask[-1], mask[:, -1], mask[..., 3] = 0.0, 0.0, 0.0    # faces that a cell of the last row or column lacks
    return x, t, mask.reshape(-1), learned.init_params(int(seed) % (1 << 31))


def _prepare_network(case, seed):
    x, t, mask, params = _network_inputs(case, seed)
    c = mdgpu.Context(9, 9, 0.0, 1.0, 0.0, 1.0)
    c.pcnet_set_params(params)
    st = dict(ctx=c, h=case["h"], w=case["w"], grad=case["grad"], x=_upload(c, x), t=_upload(c, t),
              mask=_upload(c, mask), y=c.device(x.numel(), np.float32))
    st["out"] = _tensor(st["y"])
    st["out"].zero_()
    return st


def _run_network(st):
    # the C entry points take the images where they are; the Python methods of the same names take host images
    c, L = st["ctx"], mdgpu.lib()
    if st["grad"]:
        loss = ctypes.c_double()
        rc = L.mdg_pcnet_grad(c.h, st["h"], st["w"], mdgpu.ptr(st["x"]), mdgpu.ptr(st["t"]), mdgpu.ptr(st["mask"]), 0,
                              ctypes.byref(loss))
        if rc:
            raise mdgpu.MdgError(rc, L.mdg_last_error(c.h).decode())
        return dict(loss=loss.value, grads=c.pcnet_get_params(grads=True)[1])
    rc = L.mdg_pcnet_forward(c.h, st["h"], st["w"], mdgpu.ptr(st["x"]), mdgpu.ptr(st["y"]))
    if rc:
        raise mdgpu.MdgError(rc, L.mdg_last_error(c.h).decode())
    return dict(y=st["out"])


def _exact_network(case, seed):
    x, t, mask, params = _network_inputs(case, seed)
    H, W = case["h"], case["w"]
    P = torch.as_tensor(params, device="cuda").double().requires_grad_(case["grad"])
    layers, o = [], 0
    for ci, co in LAYERS:
        layers.append((P[o:o + 9 * ci * co].reshape(9, ci, co), P[o + 9 * ci * co:o + 9 * ci * co + co]))
        o += 9 * ci * co + co

    def conv(k, a, relu=True):
        w, b = layers[k]
        h, v = a.shape[:2]
        q = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        y = b
        for i in range(9):
            y = y + (q[i // 3:i // 3 + h, i % 3:i % 3 + v].reshape(h * v, -1) @ w[i]).reshape(h, v, -1)
        return torch.relu(y) if relu else y

    def pool(a):
        h, v, ch = a.shape
        return a.reshape(h // 2, 2, v // 2, 2, ch).mean(dim=(1, 3))

    def up(a):
        return a.repeat_interleave(2, 0).repeat_interleave(2, 1)

    e0 = conv(0, x.reshape(H, W, 4).double())
    e1 = conv(1, pool(e0))
    e2 = conv(2, pool(e1))
    e3 = conv(3, pool(e2))
    d1 = conv(5, e1 + up(conv(4, e2 + up(e3))))
    y = conv(6, e0 + up(d1), relu=False)
    if not case["grad"]:
        return dict(y=torch.cat([y, torch.zeros_like(y[..., :1])], dim=2).reshape(-1))
    m = mask.reshape(H, W, 4)[..., :3].double()
    loss = 0.5 * (m * (y - t.reshape(H, W, 4)[..., :3].double()) ** 2).sum() / m.sum()
    loss.backward()
    return dict(loss=float(loss.detach()), grads=P.grad.cpu().numpy())


# --------------------------------------------------------------- the module
_KINDS = dict(markers=(_prepare_markers, _run_markers, _exact_markers), advect=(_prepare_advect, _run_advect, _exact_advect),
              rheology=(_prepare_rheology, _run_rheology, _exact_rheology), solve=(_prepare_solve, _run_solve, _exact_solve),
              energy=(_prepare_energy, _run_energy, _exact_energy),
              network=(_prepare_network, _run_network, _exact_network))


def prepare(case, seed):
    st = _KINDS[case["kind"]][0](case, seed)
    st["run"] = _KINDS[case["kind"]][1]
    torch.cuda.synchronize()            # the library works on a stream of its own
    return st


def run(state):
    return state["run"](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    k = case["kind"]
    if k == "network":
        f = sum(2.0 * (case["h"] >> s) * (case["w"] >> s) * 9 * ci * co
                for (ci, co), s in zip(LAYERS, (0, 1, 2, 3, 2, 1, 0)))
        px = case["h"] * case["w"]
        if not case["grad"]:
            return dict(bytes=32.0 * px, flops=f)
        first = 2.0 * px * 9 * 4 * 32           # no gradient is wanted for the input image
        return dict(bytes=48.0 * px, flops=3.0 * f - first)
    nx, nz = case["nx"], case["nz"]
    nc, nv = nx * nz, (nx + 1) * (nz + 1)
    nu, nw = (nx + 1) * (nz + 2), (nx + 2) * (nz + 1)
    if k == "markers":
        n = nc * case["per"] ** 2               # x, z, phase, T read; the node fields written
        s = case["stencil"]
        return dict(bytes=28.0 * n + 8.0 * (nc * (4 + case["phases"]) + 3 * nv), flops=n * (40.0 + 2 * s * 12))
    if k == "advect":
        n = nc * case["per"] ** 2               # x, z, phase, P, 3 stresses read and written, vx, vz written
        return dict(bytes=n * (2 * (8 * 6 + 4) + 16.0) + 8.0 * (6 * nc + 2 * nv + nu + nw),
                    flops=n * (4 * 60.0 + 3 * 20 + 20))
    if k == "rheology":
        nph = 2 if case["law"] == "vep" else 3
        i = 6 + nph                             # G, 3 old stresses, the laws' own fields, fractions
        b = 8.0 * ((i + 7) * (nc + nv) + 2 * nc + 2 * (nu + nw) + nu + nw + nc)
        e = 400.0 * nph
        if case["newton"]:
            b += 8.0 * (8 * nc + 4 * nv)
            e *= 9.0
        return dict(bytes=b, flops=e * (nc + nv))
    if k == "solve":
        return dict(bytes=8.0 * (nc + nv + 2 * (nu + nw + nc)), flops=60.0 * (nu + nw + nc))
    return dict(bytes=8.0 * (6 * nc + nu + nw) + 9.0 * (nx + 2) * (nz + 2), flops=40.0 * nc)


def tolerance(case):
    """About four times what the paths differ by from 64-bit sums in another
    order (exact), or between solves that stop at the same residual."""
    k = case["kind"]
    if k == "markers":      # 64-bit weights and sums; exp and log
        return {"rel": 2e-14, "max": 1e-12}
    if k == "advect":       # 64-bit arithmetic in another order
        return {"rel": 1e-15, "max": 1e-12}
    if k == "rheology":     # local iterations stop at 1e-13; the tangent divides their last bits by 1e-7
        return {"rel": 1e-6, "max": 1e-3} if case["newton"] else {"rel": 4e-13, "max": 1e-9}
    if k == "solve":        # the solver stops at a residual of 1e-8
        if case["body"] == "ellipses":      # FP64 and FP32 V-cycles: up to 3e-10 apart
            return {"rel": 4e-9, "max": 4e-7}
        return {"rel": 2e-6, "max": 1e-4}   # 4e-7 off the direct solution
    if k == "energy":       # PCG stops at a residual of 1e-8
        return {"rel": 1e-8, "max": 1e-6}
    return {"rel": 2e-2, "max": 0.5}        # bf16 operands through seven layers
