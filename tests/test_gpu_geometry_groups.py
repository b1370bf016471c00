"""Device geometry at the edges of its element groups: fewer elements than a
wave, one more or less than a wave or block, topologies interleaved in the
element list, and topologies absent."""
import numpy as np
import pytest

from oracle import orc
from tests import problems as pb
from tests.test_gpu_geometry import _device_geometry
from tests.test_gpu_geometry import ctx, nw  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


def _check(nw, ctx, coords, t, conn):
    edges = nw.mixed_edges(t, conn, coords.shape[0])
    a, v = _device_geometry(nw, ctx, coords, t, conn, edges)
    ra = orc.edge_area_vec_mixed(t, conn, coords, edges)
    rv = orc.dual_volume_mixed(t, conn, coords)
    # rounding of coordinates of order 1 in differences of one element's size
    np.testing.assert_allclose(a, ra, rtol=0, atol=1e-14 * np.abs(ra).max())
    np.testing.assert_allclose(v, rv, rtol=1e-12, atol=0)
    return a, v


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257])
def test_hex_counts_around_waves_and_blocks(nw, ctx, n):
    coords, conn = nw.hex_box(n, 1, 1, 1.0, 0.2, n)
    _check(nw, ctx, coords, np.zeros(n, np.int32), conn)


@pytest.mark.parametrize("keep", [(0, 1, 2, 3), (1, 3), (0, 2), (1,), (2, 3)])
def test_any_element_order_and_subset_of_topologies(nw, ctx, keep):
    """A shuffled element list gives the same sums in another order; subsets
    (open meshes) leave some groups empty and some nodes without volume."""
    coords, t, conn = nw.mixed_box(5, 0.5, 0.3, 0.1, seed=8)
    sel = np.flatnonzero(np.isin(t, keep))
    sel = np.random.default_rng(3).permutation(sel)
    _check(nw, ctx, coords, t[sel].copy(), conn[sel].copy())
