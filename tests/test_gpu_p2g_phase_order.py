"""Phase fractions have the same bits whatever was interpolated before them on
the same markers: first call, after a field on the same node set (whose cached
weights open the row tiles), after one on the other node set, and again; few
markers and more than the million from which the weights are worked out in the
call, a partial tile and several tiles per node row."""
import numpy as np
import pytest

import mdgpu
from test_gpu_p2g_tiles import _markers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stencil", [1, 9])
@pytest.mark.parametrize("nx,nz,per,nph", [(31, 22, 4, 3), (300, 40, 3, 9), (520, 127, 4, 2)])
def test_fractions_do_not_depend_on_earlier_calls(oracle_mod, nx, nz, per, nph, stencil):
    g, ctx, x, z, ph, rng = _markers(oracle_mod, nx, nz, per, nph)
    mat = 10.0 ** rng.uniform(-2, 2, nph)
    for centroid in (1, 0):
        def fractions():
            return np.array(ctx.p2mastah(np.zeros(2), interp_stencil=stencil, prop=1, centroid=centroid, nb_phases=nph))
        ctx.markers_set(x, z, ph)
        first = fractions()
        ctx.p2mastah(mat, centroid=centroid, interp_stencil=stencil)
        after = fractions()
        ctx.markers_set(x, z, ph)
        ctx.p2mastah(mat, centroid=1 - centroid, interp_stencil=10 - stencil)
        other = fractions()
        ctx.markers_set(x, z, ph)
        ctx.p2mastah(mat, centroid=centroid, interp_stencil=10 - stencil)
        np.testing.assert_array_equal(first, after)
        np.testing.assert_array_equal(first, other)
        np.testing.assert_array_equal(first, fractions())
