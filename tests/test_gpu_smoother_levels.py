"""The V-cycle's fused kernels (the workgroup of small levels, several smoothing
steps per launch) against the one-kernel-per-step smoothers, which apply the
same steps: smoother 1 for all levels of smoother 0 (Jacobi), the finest level
under graphs = 2 for the vertex patches of smoother 3.  Sizes lie at the edges
of both: levels of 1023, 1024 and 1056 positions, sides that leave tiles of one
row or column, long boxes, coarsening by 4.

Bound: both solves reach the tolerance on the assembled-operator residual, and
as the preconditioners differ by round-off only, the CG iterations differ by
the residual checks' granularity: 2 per outer iteration in FP64, 10% and 4 in
FP32, whose round-off perturbs CG's orthogonality (viscosity contrast 10).

One V-cycle alone is compared too, as the iteration counts would not show a
small error of the preconditioner: one outer and one CG iteration give the
velocity alpha M r and the pressure that follows from it.  There the plain side
of smoother 3 is smoother 2 with the same patch levels, none of whose kernels
the fused side runs.  Bound: the same operations in another order, some 200
smoothing steps deep: 1e-11 in FP64, 1e-4 in FP32 (the smallest levels of a
fused FP32 cycle are worked out in FP64)."""
import numpy as np
import pytest

import mdgpu

pytestmark = pytest.mark.gpu


def _problem(O, nx, nz):
    g = O.Grid(nx, nz, -0.5, 0.5, -0.5, 0.5)
    g.pure_shear(1.0)
    ctx = mdgpu.Context(nx, nz, -0.5, 0.5, -0.5, 0.5)
    ctx.set_bc(g.BCu_t, g.BCu_v, g.BCv_t, g.BCv_v, g.BCp_t, g.BCg_t)
    rng = np.random.default_rng(nx + nz)
    en = 10.0 ** rng.uniform(-0.5, 0.5, (nx - 1) * (nz - 1))
    es = 10.0 ** rng.uniform(-0.5, 0.5, nx * nz)
    neq, nm, _ = ctx.eqn_count()
    rhs = rng.standard_normal(neq)
    rhs[nm:] -= rhs[nm:].mean()
    return ctx, en, es, rhs, nm


@pytest.mark.parametrize("precision", [mdgpu.MDG_PREC_FP64, mdgpu.MDG_PREC_MIXED])
@pytest.mark.parametrize("nx,nz,patches,opts", [
    (31, 32, 0, {}), (32, 31, 0, {}), (33, 31, 0, {}), (17, 60, 0, {}), (49, 34, 0, dict(cheb_degree=7, cheb_degree_coarse=5)),
    (66, 65, 0, dict(cheb_degree=13)), (66, 65, 1, {}), (130, 25, 0, dict(coarsen4=32)), (130, 25, 1, dict(coarsen4=32)),
    (97, 83, 0, {}), (97, 83, 1, dict(cheb_degree=3, cheb_degree_coarse=9)), (150, 129, 2, dict(cheb_degree=2)),
    (257, 190, 0, dict(cheb_degree=12, cheb_degree_coarse=12)), (257, 190, 3, {}), (257, 190, 3, dict(cheb_degree=5)),
    (40, 300, 2, {})])
def test_one_cycle_matches_single_steps(oracle_mod, nx, nz, patches, opts, precision):
    ctx, en, es, rhs, nm = _problem(oracle_mod, nx, nz)
    got = []
    for s in ((3, 2) if patches else (0, 1)):
        got.append(ctx.killer_solver(2 * en, 2 * en, es, rhs[:nm], rhs[nm:], accept_diverged=True, precision=precision, smoother=s,
                                     patch_levels=patches, max_its=1, inner_max_its=1, **opts)[0])
    tol = 1e-11 if precision == mdgpu.MDG_PREC_FP64 else 1e-4
    for a, b in ((got[0][:nm], got[1][:nm]), (got[0][nm:], got[1][nm:])):
        assert np.linalg.norm(b) > 0
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("precision", [mdgpu.MDG_PREC_FP64, mdgpu.MDG_PREC_MIXED])
@pytest.mark.parametrize("fused,plain", [(dict(smoother=0), dict(smoother=1)),
                                         (dict(smoother=3), dict(smoother=3, graphs=2))])
@pytest.mark.parametrize("nx,nz,opts", [
    (31, 32, {}), (32, 31, {}), (33, 31, {}), (17, 60, {}), (49, 34, dict(cheb_degree=7, cheb_degree_coarse=5)),
    (66, 65, dict(graphs=1)), (130, 25, dict(coarsen4=32)), (97, 83, dict(graphs=0)), (150, 129, dict(cheb_degree=2)),
    (257, 190, dict(cheb_degree=12, cheb_degree_coarse=12))])
def test_fused_levels_match_single_steps(oracle_mod, nx, nz, opts, fused, plain, precision):
    ctx, en, es, rhs, nm = _problem(oracle_mod, nx, nz)
    tol = 1e-9 if precision == mdgpu.MDG_PREC_FP64 else 1e-6
    its = []
    for s in (fused, plain):
        sol, o = ctx.killer_solver(2 * en, 2 * en, es, rhs[:nm], rhs[nm:], rel_tol=tol, precision=precision, **{**opts, **s})
        r = rhs - ctx.stokes_apply(2 * en, 2 * en, es, sol)
        assert np.linalg.norm(r) <= 1.01 * tol * np.linalg.norm(rhs)
        its.append((o.its, o.inner_its))
    assert abs(its[0][0] - its[1][0]) <= 1, its
    slack = 2 * its[1][0] + (0 if precision == mdgpu.MDG_PREC_FP64 else 0.1 * its[1][1] + 4)
    assert abs(its[0][1] - its[1][1]) <= slack, its
