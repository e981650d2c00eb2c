"""Grid rheology and Newton tangent over the stress exponents that take their
own branch (1, 2 and 3 as products, others through pow), prefactors with and
without pressure dependence, node-wise friction and dilation angles, on node
counts that leave a partial wavefront, against the oracle.

Tolerance: the local iterations stop at a 1e-13 relative residual and the
return map at |F| < 1e-12, so fields agree to 1e-10 of their largest value
(a product and pow differ by ulps).  The tangent divides by twice a relative
perturbation of 1e-5 (centres) or 1e-7 (vertices) of a strain rate or pressure
of order 0.1 or more: 1e-12 / 2e-6 and 1e-13 n / 2e-8 of the viscosity, below
1e-6 and 2e-5 of the larger of the row and the viscosity row."""
import numpy as np
import pytest

import mdgpu
from test_gpu_rheology import _ctx, _fields, _phase_pair

pytestmark = pytest.mark.gpu


def _phases(O, n_pwl, n_lin, V):
    return [_phase_pair(O, d) for d in (
        dict(pwlv=1, n_pwl=n_pwl, A_pwl=0.5, F_pwl=0.8, V_pwl=V, Q_pwl=1.0, linv=1, F_lin=0.7, A_lin=2.5, n_lin=n_lin,
             m_lin=2.0, Q_lin=1.5, V_lin=V, gs_ref=0.7),
        dict(pwlv=1, n_pwl=n_pwl, A_pwl=2.0, Q_pwl=0.5, plast=1, C=0.8, fric=0.5, dil=0.1, eta_vp=0.05, beta=20.0))]


@pytest.mark.parametrize("nx,nz", [(3, 4), (37, 29)])
@pytest.mark.parametrize("n_pwl,n_lin,V", [(1.0, 1.0, 0.0), (2.0, 3.0, 0.1), (3.0, 2.0, 0.0), (3.3, 1.7, 0.1)])
def test_exponents_match_oracle(oracle_mod, n_pwl, n_lin, V, nx, nz):
    O = oracle_mod
    g, ctx = _ctx(O, nx, nz)
    pairs = _phases(O, n_pwl, n_lin, V)
    common = dict(step=3, elastic=1, dt=0.5, R=1.0, zeroC=0.6, min_eta=1e-3, max_eta=1e3, eta_tol=1e-12, Tiimin=1e-3,
                  scale_E=1.0, scale_eta=1.0, d_min=1e-3)
    md, prm = O.OrcRheoModel(**common), mdgpu.RheoParams(average=0, **common)
    for centroid in (1, 0):
        n = ctx.node_count(centroid)
        f, rng = _fields(n, 2, seed=5 + centroid)
        f["d"] = rng.uniform(0.3, 1.5, n)
        f["fric"], f["dil"] = rng.uniform(0.1, 0.6, n), rng.uniform(0.0, 0.2, n)
        tag = g.BCp_t if centroid else g.BCg_t
        args = [f[k] for k in ("perc", "G", "T", "P", "exx", "ezz", "exz", "sxx0", "szz0", "sxz0")]
        node = dict(fric=f["fric"], dil=f["dil"], d=f["d"], tag=tag, centroid=centroid)
        ref = O.rheology_nodes(md, [p[0] for p in pairs], *args, **node, average=0)
        out = ctx.viscosity_grid([p[1] for p in pairs], prm, centroid, **f)
        for k in mdgpu.RHEO_OUT:
            np.testing.assert_allclose(out[k], ref[k], rtol=1e-10, atol=1e-10 * np.abs(ref[k]).max() + 1e-300, err_msg=k)
        D_o = O.tangent_nodes(md, [p[0] for p in pairs], *args, **node)
        D_g = ctx.tangent_grid([p[1] for p in pairs], prm, centroid, **f)
        visc = np.abs(D_o[0 if centroid else 2]).max()
        for r in range(D_o.shape[0]):
            np.testing.assert_allclose(D_g[r], D_o[r], rtol=0, err_msg="row %d" % r,
                                       atol=(1e-6 if centroid else 2e-5) * max(np.abs(D_o[r]).max(), visc))
