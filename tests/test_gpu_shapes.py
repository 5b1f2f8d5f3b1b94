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


@pytest.mark.parametrize("model,nmol,chunks,path,precision", [
    ("TIP4P", 256, 1, 0, 0),     # whole ring: 255 partners a lane, the last mask word one bit short
    ("TIP5P", 300, 7, 0, 0),     # 5-site records (narrow last plane), ragged chunks
    ("TIP3P", 301, 64, 0, 0),    # more chunks than a screening batch has partners
    ("TIP4P", 256, 3, 0, 1),     # FP64 records: eight planes of two words
    ("TIP4P", 300, 1, 3, 0),     # split-global
    ("TIP5P", 300, 4, 2, 0),     # global-state path
    ("TIP4P", 1000, 1, 2, 0),    # global-state path, window beyond one word
])
def test_screened_pairs_match_oracle(model, nmol, chunks, path, precision):
    """Step-0 forces of bulk water where the screening masks, their tails and
    the record planes meet an edge.  FP32 pair math: 1e-5 relative RMS (a
    force is a sum of about 100 pairs rounded at 6e-8 each, against terms up
    to 50 times the sum); FP64: 1e-11."""
    from helpers import oracle_for, rel_rms
    from remd_amd import inputs

    L = max((nmol * 29.9) ** (1.0 / 3.0), 19.2)
    s = inputs.config_bulk(seed=11, nmol=nmol, L=L, ntemp=1, npress=1, model=model) if nmol <= 343 else None
    if s is None:
        s = inputs.config_bulk(seed=11, nmol=343, L=L, ntemp=1, npress=1, model=model)
        rng = np.random.RandomState(11)
        s.nmol = nmol
        s.states = inputs._states(rng, inputs.molecule(model), inputs.place_lattice(nmol, L), s.T, (L, L, L), 0.5, 0.05)
    o = oracle_for(s)
    o.initialize_property()
    g = ra.REMDGPU(s, precision=precision, chunks=chunks, path=path)
    assert rel_rms(g.state(0)["f"], o.state()["f"]) < (1e-11 if precision else 1e-5)
    assert rel_rms(g.state(0)["n"], o.state()["n"]) < (1e-11 if precision else 1e-5)


@pytest.mark.parametrize("R", [10.3, 10.6])
def test_tube_screening_rule(R):
    """Step-0 forces either side of the radius from which tubes screen their
    partners (same tolerance)."""
    from helpers import oracle_for, rel_rms
    from remd_amd import inputs

    s = inputs.config_tube(seed=13, nmol=150, R=R, Lz=30.0, ntemp=1, npress=1, nfwall=500, r_acc=R - 2.8)
    o = oracle_for(s)
    o.initialize_property()
    g = ra.REMDGPU(s)
    assert rel_rms(g.state(0)["f"], o.state()["f"]) < 1e-5
