"""The row tiles of the marker -> grid kernels at their edges against the
oracle: boxes one node narrower and wider than a tile, high enough for four
node rows per block and one row below, phase tables at the length that stays
in LDS, one and the most phases, and phase fractions before and after the
cached weights exist (a million markers have them worked out in the call).

Tolerance: a node sums the same weights and products as the oracle in another
order, all weights positive: (markers per node) ulps, below 1e-13; fields pass
one exp or division more, 1e-12 as in the other marker -> grid tests."""
import numpy as np
import pytest

import mdgpu
from mdgpu import setups as S

pytestmark = pytest.mark.gpu


def _markers(O, nx, nz, per, nph):
    g = O.Grid(nx, nz, -0.5, 0.5, -0.3, 0.45)
    x, z = S.put_markers(g.xg, g.zg, g.dx, g.dz, per, per, seed=nx)
    rng = np.random.default_rng(nz)
    ph = rng.integers(0, nph, x.size).astype(np.int32)
    ph[::97] = -1
    ctx = mdgpu.Context(nx, nz, -0.5, 0.5, -0.3, 0.45)
    ctx.markers_set(x, z, ph)
    return g, ctx, x, z, ph, rng


@pytest.mark.parametrize("stencil", [1, 9])
@pytest.mark.parametrize("nx,nz,per,nph", [(256, 9, 2, 1), (257, 7, 3, 9), (258, 6, 2, 32), (3, 2047, 2, 2), (4, 2048, 2, 3),
                                           (262, 257, 4, 5)])
def test_phase_fractions_and_tables(oracle_mod, nx, nz, per, nph, stencil):
    g, ctx, x, z, ph, rng = _markers(oracle_mod, nx, nz, per, nph)
    for centroid in (1, 0):
        kw = dict(prop=1, centroid=centroid, nb_phases=nph)
        ref = oracle_mod.p2mastah(g, x, z, ph, np.zeros(2), stencil=stencil, **kw)
        tags = np.full(ref.shape[1], -1, np.int8)
        tags[2:5] = 30
        for _ in range(2):      # general path or, with many markers, tiles; then tiles
            got = ctx.p2mastah(np.zeros(2), interp_stencil=stencil, **kw)
            np.testing.assert_allclose(np.array(got), ref, rtol=1e-13, atol=1e-15)
            for n_tab, avg in ((nph, 0), (64, 1), (65, 2)):
                tab = 10.0 ** rng.uniform(-2, 2, n_tab if n_tab >= nph else nph)
                r = oracle_mod.p2mastah(g, x, z, ph, tab, avg=avg, centroid=centroid, stencil=stencil)
                f = ctx.p2mastah(tab, avg=avg, centroid=centroid, interp_stencil=stencil)
                np.testing.assert_allclose(f, r, rtol=1e-12)
        ref = oracle_mod.p2mastah(g, x, z, ph, np.zeros(2), stencil=stencil, node_type=tags, **kw)
        got = ctx.p2mastah(np.zeros(2), interp_stencil=stencil, node_type=tags, **kw)
        np.testing.assert_allclose(np.array(got), ref, rtol=1e-13, atol=1e-14)
