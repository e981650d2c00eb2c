"""The marker kernels where their divisions leave the fast path, and with
tagged vertices, against the oracle bit for bit: boxes whose cell widths lie
beyond exact_div's divisors, boxes far from and around the origin, markers
at subnormal coordinates, velocities that are zero, signed zero or tiny, and
vertices tagged 31 (the tag-reading instantiations of the grid -> marker
kernels)."""
import numpy as np
import pytest

import mdgpu
from mdgpu import setups as S

pytestmark = pytest.mark.gpu

BOXES = {"unit": (0.0, 1.0, -1.0, 0.0), "centred": (-3.0, 3.0, -3.0, 3.0), "tiny": (0.0, 1e-60, 0.0, 1e-60),
         "huge": (-1e60, 1e60, 0.0, 2e60), "far": (1e7, 1e7 + 1.0, -1e7, -1e7 + 1.0)}


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def _box(O, name, n=21):
    b = BOXES[name]
    g = O.Grid(n + 1, n + 1, *b)
    g.pure_shear(0.0)
    x, z = S.put_markers(g.xg, g.zg, g.dx, g.dz, 3, 3, seed=4, noise=name != "centred")
    x[:6] = [b[0], b[1], 0.5 * (b[0] + b[1]), g.xg[3], g.xvz[4], 5e-324 if b[0] <= 0 <= b[1] else b[0]]
    z[:6] = [b[2], b[3], 0.5 * (b[2] + b[3]), g.zg[5], g.zvx[2], 1e-310 if b[2] <= 0 <= b[3] else b[3]]
    ph = np.zeros(x.size, np.int32)
    ph[7::50] = -1
    ctx = mdgpu.Context(n + 1, n + 1, *b)
    return g, ctx, x, z, ph


@pytest.mark.parametrize("flow", ["random", "rest", "tiny"])
@pytest.mark.parametrize("name", list(BOXES))
def test_velocities_and_rk4(oracle_mod, name, flow):
    O = oracle_mod
    g, ctx, x, z, ph = _box(O, name)
    ctx.set_bc(g.BCu_t, g.BCu_v, g.BCv_t, g.BCv_v, g.BCp_t, g.BCg_t)
    rng = np.random.default_rng(8)
    s = {"random": 1.0, "rest": 0.0, "tiny": 1e-300}[flow]
    u, v = rng.standard_normal(g.BCu_t.size) * s, rng.standard_normal(g.BCv_t.size) * s   # rest: +0 and -0
    u[::3] *= 0.0
    for conserv in (0, 1):
        got, ref = ctx.v2p(u, v, x, z, ph, conserv=conserv), O.v2p(g, u, v, x, z, ph, conserv=conserv)
        for a, b in zip(got, ref):
            assert np.array_equal(_bits(a), _bits(b))
        dt = 0.4 * g.dx
        r = O.advect_rk4(g, u, v, dt, x, z, ph, conserv=conserv, vx=np.zeros(x.size), vz=np.zeros(x.size))
        a = [x.copy(), z.copy(), ph.copy(), np.zeros(x.size), np.zeros(x.size)]
        ctx.advect_rk4(u, v, dt, a[0], a[1], a[2], conserv=conserv, vx=a[3], vz=a[4])
        assert np.array_equal(a[2], r[2])
        for q in (0, 1, 3, 4):
            assert np.array_equal(_bits(a[q]), _bits(r[q])), (conserv, q)


@pytest.mark.parametrize("tagged", [False, True])
@pytest.mark.parametrize("name", list(BOXES))
def test_grid_to_markers(oracle_mod, name, tagged):
    O = oracle_mod
    g, ctx, x, z, ph = _box(O, name)
    if tagged:
        g.BCg_t[-5 * g.Nx:] = 31
    ctx.set_bc(g.BCu_t, g.BCu_v, g.BCv_t, g.BCv_v, g.BCp_t, g.BCg_t)
    rng = np.random.default_rng(9)
    nc, nv = g.BCp_t.size, g.BCg_t.size
    F, G = rng.standard_normal(nc), rng.standard_normal(nv)
    assert np.array_equal(_bits(ctx.g2p_centroids(F, x, z, ph)), _bits(O.g2p_centroids(g, F, x, z, ph)))
    assert np.array_equal(_bits(ctx.g2p_vertices(G, x, z, ph)), _bits(O.g2p_vertices(g, G, x, z, ph)))
    grids = [rng.standard_normal(m) for m in (nc, nc, nv, nc, nc, nv)]
    m = [rng.standard_normal(x.size) for _ in range(3)]
    ref = O.update_particle_stress(g, *grids, x, z, ph, *[a.copy() for a in m])
    got = [a.copy() for a in m]
    ctx.update_particle_stress(*grids, x, z, ph, *got)
    for a, b in zip(got, ref):
        assert np.array_equal(_bits(a), _bits(b))


def test_tags_of_a_refused_set_bc(oracle_mod):
    """A set_bc that is refused for its last array has replaced the centre tags
    all the same: the grid -> marker kernels read them."""
    O = oracle_mod
    g, ctx, x, z, ph = _box(O, "unit")
    ctx.set_bc(g.BCu_t, g.BCu_v, g.BCv_t, g.BCv_v, g.BCp_t, g.BCg_t)
    g.BCp_t[-4 * (g.Nx - 1):] = 30
    arrays = [np.ascontiguousarray(a) for a in (g.BCu_t, g.BCu_v, g.BCv_t, g.BCv_v, g.BCp_t)]
    assert ctx._L.mdg_set_bc(ctx.h, *[mdgpu.ptr(a) for a in arrays], None) != 0
    F = np.random.default_rng(10).standard_normal(g.BCp_t.size)
    assert np.array_equal(_bits(ctx.g2p_centroids(F, x, z, ph)), _bits(O.g2p_centroids(g, F, x, z, ph)))
