"""Two contexts used from two threads at once give what each gives alone: Stokes
solves whose small levels need different amounts of LDS, and phase fractions of
many phases, which need different amounts too.  Kernel attributes belong to the
process, so what one call asks for must not depend on the other's."""
import threading

import numpy as np
import pytest

import mdgpu
from test_gpu_p2g_tiles import _markers

pytestmark = pytest.mark.gpu


def _solver(O, nx, nz, precision):
    g = O.Grid(nx, nz, -0.5, 0.5, -0.5, 0.5)
    g.pure_shear(1.0)
    ctx = mdgpu.Context(nx, nz, -0.5, 0.5, -0.5, 0.5)
    ctx.set_bc(g.BCu_t, g.BCu_v, g.BCv_t, g.BCv_v, g.BCp_t, g.BCg_t)
    rng = np.random.default_rng(nx * nz)
    en = 10.0 ** rng.uniform(-0.5, 0.5, (nx - 1) * (nz - 1))
    es = 10.0 ** rng.uniform(-0.5, 0.5, nx * nz)
    neq, nm, _ = ctx.eqn_count()
    rhs = rng.standard_normal(neq)
    rhs[nm:] -= rhs[nm:].mean()
    return lambda: ctx.killer_solver(2 * en, 2 * en, es, rhs[:nm], rhs[nm:], rel_tol=1e-6, precision=precision)[0]


def _fractions(O, nx, nz, nph, stencil):
    _, ctx, x, z, ph, _ = _markers(O, nx, nz, 3, nph)
    ctx.p2mastah(np.ones(nph))      # cached weights: row tiles
    return lambda: np.array(ctx.p2mastah(np.zeros(2), interp_stencil=stencil, prop=1, centroid=1, nb_phases=nph))


def _together(calls, reps):
    alone = [f() for f in calls]
    errors = []

    def work(q):
        try:
            for _ in range(reps):
                np.testing.assert_array_equal(calls[q](), alone[q])
        except BaseException as e:      # noqa: BLE001 (reported by the main thread)
            errors.append((q, e))
    threads = [threading.Thread(target=work, args=(q,)) for q in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("precision", [mdgpu.MDG_PREC_FP64, mdgpu.MDG_PREC_MIXED])
def test_solves(oracle_mod, precision):
    _together([_solver(oracle_mod, 31, 32, precision), _solver(oracle_mod, 12, 11, precision)], 8)


@pytest.mark.parametrize("stencil", [1, 9])
def test_phase_fractions(oracle_mod, stencil):
    _together([_fractions(oracle_mod, 70, 41, 32, stencil), _fractions(oracle_mod, 50, 33, 21, stencil)], 40)
