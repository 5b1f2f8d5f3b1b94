"""GPU kernels at the sizes where their tiling can go wrong, against the
oracle."""
import numpy as np
import pytest

import pyoracle as po
import remd_amd as ra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfw", [3, 4, 5, 7, 1003])
def test_wall_table_tube_node_counts(nfw):
    """Tables whose node count is below, at and beside the nodes of one
    workgroup (4).  The same operations in the same order as the oracle's,
    so 1e-12 of the largest entry, as for the other tables."""
    g = ra.wall_table(1, nfw, 9.0, 3.277, 0.3886, 0.38016)
    o = po.wall_table_tube(nfw, 9.0, 3.277, 0.3886, 0.38016)
    assert np.allclose(g, o, rtol=1e-12, atol=1e-12 * np.max(np.abs(o)))
