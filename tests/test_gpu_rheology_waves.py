"""Grid rheology and Newton tangent do not depend on which nodes share a
wavefront: the bits of a node's results are those it has in a wave filled with
its own state, when waves hold 64 random states and when they hold two.  The
laws that a phase has are tested inside the local iterations, and lanes that
leave those at different trips must not change a test's outcome for the others.

Two sets of states: mixed ones (strain rates over three decades, temperatures
on both sides of the Peierls limit, nodes without one or the other phase), and
ones at the limit of their stopping test, whose strain rate is set (by
bisection of the trips of the same iteration on the host) so that round-off
decides whether a state takes one trip more at its base value or at a
perturbed one of the tangent's differences."""
import numpy as np
import pytest

import mdgpu
from test_gpu_rheology import LAWS, _ctx, _phase_pair

pytestmark = pytest.mark.gpu
WAVE, STATES = 64, 512
CREEP = dict(cstv=0, pwlv=1, n_pwl=3.0, A_pwl=0.5, F_pwl=0.8, Q_pwl=1.0, linv=1, A_lin=2.5, F_lin=0.7, n_lin=1.0, Q_lin=1.5,
             gs_ref=1.0)
DT = 0.5


def _mixed(rng):
    s = 10.0 ** rng.uniform(-2, 1, STATES)
    perc = rng.dirichlet(np.ones(len(LAWS)), STATES).T.copy()
    perc[0, ::5] = 0.0
    perc[1, 1::7] = 0.0
    perc[2, 2::3] = 0.0
    perc[1, perc.sum(0) == 0] = 1.0
    f = dict(perc=perc, G=rng.uniform(0.5, 2.0, STATES), T=rng.uniform(0.7, 1.3, STATES), P=rng.uniform(0.0, 3.0, STATES),
             d=rng.uniform(0.3, 1.5, STATES), phi=rng.uniform(0, 0.05, STATES))
    f["phi"][::4] = 0.0
    for k in ("exx", "ezz", "exz"):
        f[k] = s * rng.normal(0, 1, STATES)
    for k in ("sxx0", "szz0", "sxz0"):
        f[k] = s * rng.normal(0, 0.3, STATES)
    return f


def _trips(f, s):
    """Local iterations of CREEP at the strain rates times s."""
    exx, ezz, exz = (s * f[k] for k in ("exx", "ezz", "exz"))
    E = np.sqrt(0.5 * (exx ** 2 + ezz ** 2 + (exx + ezz) ** 2) + exz ** 2)
    B = 0.8 * 0.5 ** (-1.0 / 3.0) * np.exp(1.0 / 3.0 / f["T"])
    Bl = 0.7 / 2.5 * np.exp(1.5 / f["T"])
    el = f["G"] * DT
    eta = np.minimum(np.minimum(B * E ** (1.0 / 3.0 - 1.0), el), Bl)
    n = np.zeros(E.size, int)
    run = np.ones(E.size, bool)
    for it in range(20):
        T = 2.0 * eta * E
        ep, el_ = (2.0 * B) ** -3.0 * T ** 3, T / (2.0 * Bl)
        r = E - T / (2.0 * el) - ep - el_
        n[run] += 1
        run &= ~(np.abs(r / E) < 1e-13)
        eta = np.where(run, eta - r / (-E / el - el_ / eta - 3.0 * ep / eta), eta)
    return n


def _at_the_limit(rng):
    f = dict(G=rng.uniform(0.5, 2.0, STATES), T=rng.uniform(0.7, 1.3, STATES), P=rng.uniform(0.0, 3.0, STATES))
    for k in ("exx", "ezz", "exz"):
        f[k] = rng.normal(0, 1, STATES)
    lo, hi = np.full(STATES, 0.02), np.full(STATES, 10.0)
    k = 4       # trips: at most k at lo, more at hi
    ok = (_trips(f, lo) <= k) & (_trips(f, hi) > k)
    for _ in range(60):
        mid = np.sqrt(lo * hi)
        more = _trips(f, mid) > k
        lo, hi = np.where(more, lo, mid), np.where(more, mid, hi)
    assert ok.sum() > STATES // 4
    use = rng.choice(np.flatnonzero(ok), STATES)
    f = {q: v[use] for q, v in f.items()}
    for q in ("exx", "ezz", "exz"):
        f[q] = lo[use] * f[q]
    return dict(f, perc=np.ones((1, STATES)))


@pytest.mark.parametrize("average", [0, 1, 2])
@pytest.mark.parametrize("laws", [(0, 1, 2), (1, 2, 0), (2, 0, 1), None])
@pytest.mark.parametrize("centroid", [1, 0])
def test_same_bits_for_any_neighbours(oracle_mod, centroid, laws, average):
    g, ctx = _ctx(oracle_mod, 256 + centroid, 128 + centroid)
    n = ctx.node_count(centroid)
    assert n == WAVE * STATES
    prm = mdgpu.RheoParams(step=3, elastic=1, average=average, dt=DT, R=1.0, zeroC=0.6, min_eta=1e-6, max_eta=1e6, eta_tol=1e-12,
                           Tiimin=1e-6, scale_E=1.0, scale_eta=1.0, T_peierls=1.0, d_min=1e-3)
    phases = [_phase_pair(oracle_mod, d)[1] for d in ([LAWS[q] for q in laws] if laws else [CREEP])]
    rng = np.random.default_rng(11 + centroid)
    f = _mixed(rng) if laws else _at_the_limit(rng)
    wave = np.arange(n) // WAVE
    pair = rng.integers(0, STATES, (STATES, 2))[wave, rng.integers(0, 2, n)]
    alone = None
    for state in (wave, rng.integers(0, STATES, n), pair):
        a = {k: np.ascontiguousarray(v[..., state]) for k, v in f.items()}
        got = {k: v for k, v in ctx.viscosity_grid(phases, prm, centroid, **a).items() if k in mdgpu.RHEO_OUT}
        D = ctx.tangent_grid(phases, prm, centroid, **a)
        assert np.isfinite(D).all()
        got.update({"D%d" % r: D[r] for r in range(D.shape[0])})
        if alone is None:
            alone = {k: v[::WAVE] for k, v in got.items()}
        for k, v in got.items():
            np.testing.assert_array_equal(v, alone[k][state], err_msg=k)
