"""GPU kernels at the sizes where their tiling can go wrong, against the
oracle."""
import numpy as np
import pytest

import pyoracle as po
import remd_amd as ra

pytestmark = pytest.mark.gpu


def _bulk(nmol, model, nrep=2, seed=17):
    from remd_amd import inputs

    L = max((nmol * 29.9) ** (1.0 / 3.0), 19.2)
    s = inputs.config_bulk(seed=seed, nmol=nmol, L=L, ntemp=nrep, npress=1, model=model) if nmol <= 343 else None
    if s is None:
        s = inputs.config_bulk(seed=seed, nmol=343, L=L, ntemp=nrep, npress=1, model=model)
        rng = np.random.RandomState(seed)
        s.nmol = nmol
        s.states = inputs._states(rng, inputs.molecule(model), inputs.place_lattice(nmol, L), s.T, (L, L, L), 0.5, 0.05)
    s.pconstant = 1
    s.dt_fs = 0.2  # unrelaxed contacts
    s.interval = 12  # two sorts
    return s


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
    s = _bulk(nmol, model, nrep=1, seed=11)
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


@pytest.mark.parametrize("model,nmol,chunks,precision,abort", [
    ("TIP4P", 513, 1, 0, False),   # ragged parts
    ("TIP3P", 600, 4, 0, False),   # butterfly over chunks
    ("TIP5P", 700, 2, 1, False),   # FP64
    ("TIP4P", 2100, 1, 1, False),  # site records in global memory, one copy per part
    ("TIP4P", 600, 1, 0, True),    # parts that give up: completed by one workgroup per replica
])
def test_global_path_parts_keep_the_bits(model, nmol, chunks, precision, abort, monkeypatch):
    """A global-state job alone is split over workgroups, in a batch it is
    not: the same bits, also when the split launch gives up."""
    s = _bulk(nmol, model)
    a = ra.REMDGPU(s, precision=precision, chunks=chunks, path=ra.PATH_GLOBAL)
    b = ra.REMDGPU(s, precision=precision, chunks=chunks, path=ra.PATH_GLOBAL)
    if abort:
        monkeypatch.setenv("REMD_GLOBAL_ABORT", "1")
    a.execute_steps(s.T, s.P)
    monkeypatch.delenv("REMD_GLOBAL_ABORT", raising=False)
    if not abort:
        assert a.launch_path()[1] > 1
    bt = ra.Batch()
    bt.add(b)
    b.set_conditions(s.T, s.P)
    bt.execute()
    assert np.array_equal(a.all_averages(), b.all_averages())
    for r in range(s.nreplica):
        x, y = a.state(r), b.state(r)
        for k in ("r", "v", "f", "q", "p", "n", "id", "scal"):
            assert np.array_equal(x[k], y[k]), k
    bt.close()


@pytest.mark.parametrize("path", [2, 3])
def test_replica_gone_non_finite_has_no_pairs(path):
    """A replica whose positions are not numbers has no partner inside the
    cutoff: forces, torques and energies are exactly zero, and the replica
    beside it keeps its forces (1e-5 relative RMS, as above)."""
    from helpers import oracle_for, rel_rms

    s = _bulk(800, "TIP4P", nrep=2)
    good = s.states[0].r
    s.states[1].r = np.full_like(good, np.nan)
    g = ra.REMDGPU(s, path=path)
    bad = g.state(1)
    assert np.all(bad["f"] == 0.0) and np.all(bad["n"] == 0.0)
    assert np.all(g.averages(1)[:3] == 0.0)
    o = oracle_for(s, 0)
    o.initialize_property()
    assert rel_rms(g.state(0)["f"], o.state()["f"]) < 1e-5


@pytest.mark.parametrize("nmol,path,keys", [
    (4, 0, "spread"), (63, 0, "spread"), (257, 0, "spread"),
    (515, 3, "spread"),
    (300, 0, "equal"),     # one bucket holds every key
    (300, 0, "layers"),    # equal keys in a few buckets, some zeros of either sign
    (300, 0, "outside"),   # keys below 0 and above 1: the outer buckets
    (300, 0, "nan"),       # a key without a place in the searches
])
def test_bucket_sort_order_and_windows(nmol, path, keys, monkeypatch):
    """The bucket sort gives the stable order of the sort coordinate, and the
    windows the counting sort gives (except where a NaN leaves that sort
    without an order)."""
    s = _bulk(nmol, "TIP4P", nrep=1)
    rng = np.random.RandomState(nmol)
    z = rng.permutation(s.states[0].r[:, 2] + 0.3 / nmol * rng.rand(nmol))
    if keys == "equal":
        z[:] = 0.37
    elif keys == "layers":
        z = rng.randint(0, 5, nmol) / 5.0
        z[z == 0.0] = np.where(rng.rand(int((z == 0.0).sum())) < 0.5, -0.0, 0.0)
    elif keys == "outside":
        z = 3.0 * z - 1.0
    elif keys == "nan":
        z[7] = np.nan
    s.states[0].r[:, 2] = z
    got = []
    for least in (1, 10 ** 6):
        monkeypatch.setenv("REMD_SORT_RADIX_MIN", str(least))
        g = ra.REMDGPU(s, path=path)
        g.set_debug(True)
        g.compute_forces(True)
        got.append((g.state(0)["id"], g.window(0, with_full=True)))
    assert np.array_equal(got[0][0], np.argsort(z, kind="stable"))
    if keys != "nan":
        assert np.array_equal(got[1][0], got[0][0])
        for a, b in zip(got[0][1], got[1][1]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("nmol,precision,keys", [
    (65, 0, "spread"), (515, 0, "spread"), (700, 1, "spread"),
    (300, 0, "outside"),    # keys below zero come last in this path's order
    (300, 0, "nan"),
    (1100, 1, "spread"),    # records in global memory: the radix sort
])
def test_global_path_sort_order_and_windows(nmol, precision, keys):
    """The global-state path's order is that of the keys' bits as unsigned
    integers, stable; its windows those of the split-global path."""
    s = _bulk(nmol, "TIP4P", nrep=1)
    rng = np.random.RandomState(nmol)
    z = rng.permutation(s.states[0].r[:, 2] + 0.3 / nmol * rng.rand(nmol))
    if keys == "outside":
        z = 3.0 * z - 1.0
    elif keys == "nan":
        z[7] = np.nan
    s.states[0].r[:, 2] = z
    got = []
    for path, prec in ((ra.PATH_GLOBAL, precision), (ra.PATH_SPLIT, 0)):
        g = ra.REMDGPU(s, precision=prec, path=path)
        g.set_debug(True)
        g.compute_forces(True)
        got.append((g.state(0)["id"], g.window(0, with_full=True)))
    assert np.array_equal(got[0][0], np.argsort((z + 0.0).view(np.uint64), kind="stable"))
    if keys == "spread":
        assert np.array_equal(got[1][0], got[0][0])
        for a, b in zip(got[0][1], got[1][1]):
            assert np.array_equal(a, b)
