"""The first and last passes of a run where their sizes change: grids whose
points are no multiple of four, fewer points than a workgroup, several
workgroups; bucket counts on both sides of the one-workgroup scan's two sizes
and of the scan by tiles.  Results equal the oracle's; the run's sums equal
those of what it returns."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu


def _bits(a):
    a = np.ascontiguousarray(a, np.float32).ravel()
    return np.where(np.isnan(a), np.float32(np.nan), a).view(np.uint32)


def _block(n):
    p = synthetic.uniform(n, seed=n)
    return ingest.make_block(p, n, (0, 0, 0), (1, 1, 1))


def _check_stats(st, s, npts, density):
    for code, key in enumerate(("cells_scan", "cells_cic", "cells_incomplete", "cells_outside",
                                "cells_degenerate")):
        assert st[key] == int((s == code).sum())
    assert st["points_deposited"] + st["points_offblock"] == int(npts[s <= 1].sum())
    d = np.ascontiguousarray(density, np.float32).ravel()
    assert st["max_dense"] == d.max()
    # tot_mass is the float64 sum times the (float32) cell size; two orders of
    # addition of n positive numbers differ by at most n 2^-52
    ratio = st["tot_mass"] / d.astype(np.float64).sum()
    assert abs(ratio / float(np.float32(ratio)) - 1.0) <= (d.size + 2) * 2.0 ** -52


@pytest.mark.parametrize("g", [(2, 2, 2), (3, 3, 3), (11, 9, 7), (33, 32, 31), (65, 63, 61)])
@pytest.mark.parametrize("n", [700, 3300])
def test_scan_ends(oracle, n, g):
    print("run ends scan", n, g, flush=True)
    hb = _block(n)
    run = D.StagedRun([hb])
    want = oracle.dense_single(oracle.Block.from_host(hb), g)
    for _ in range(2):             # a run after a run: nothing is left of the first
        run.run(g)
        st = run.sync()
        d = run.fetch(0)["density"]
        s, npts = run.cells(0)
        assert np.array_equal(s, want["status"]) and np.array_equal(npts, want["npts"])
        assert np.array_equal(_bits(d), _bits(want["density"]))
        _check_stats(st, s, npts, d)


@pytest.mark.parametrize("n", [900, 4500, 15000, 19000])
def test_exact_ends(oracle, n):
    print("run ends exact", n, flush=True)
    hb, g = _block(n), (21, 17, 13)
    run = D.StagedRun([hb])
    want = oracle.exact_dense(oracle.Block.from_host(hb), g)
    for _ in range(2):
        run.run(g, assignment=D.EXACT_VORONOI, precision=D.FP64)
        run.sync()
        assert np.array_equal(run.owner(0), want["owner"])
        s, npts = run.cells(0)
        assert np.array_equal(s, want["status"]) and np.array_equal(npts, want["npts"])
