"""The geometry and scan kernels over all cells (cells_geom.hip, cells_scan.hip:
the automatic choice for several blocks and for 16384 cells and more) against
the oracle, through the C ABI: statuses, counts, volumes and densities bit for
bit where their tiles of 64 cells end, where stars exceed the geometry
kernel's tables, on degenerate cells, with boxes of every class (tiles, one
wave per cell by lines, one wave by probes) and at the eps the verdict
shortcut stops at.  The other multi-block tests run them too."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu


def _bits(a):
    a = np.ascontiguousarray(a, np.float32).ravel()
    u = a.view(np.uint32).copy()
    u[np.isnan(a)] = 0x7FC00000
    return u


@pytest.fixture(scope="module")
def blocks():
    out = {}
    out["uniform"] = ingest.periodic_block(synthetic.uniform(16385, seed=61), 4.0 / 25.4)
    p64 = synthetic.jittered_lattice64(26, 1e-6, seed=4)
    out["jitter"] = ingest.periodic_block(synthetic.jittered_lattice(26, 1e-6, seed=4), 3.0 / 26,
                                          p64=synthetic.lattice_tiebreak(p64, 26))
    return out


@pytest.mark.parametrize("name,g,eps", [
    ("uniform", (50, 50, 50), 1e-4), ("uniform", (12, 9, 10), 1e-4),
    ("uniform", (400, 37, 64), 1e-4),      # lines of more than 16 points
    ("uniform", (900, 24, 24), 1e-4),      # and of more than 32
    ("uniform", (40, 40, 40), 0.0), ("uniform", (40, 40, 40), -1e-5),
    ("jitter", (60, 60, 60), 1e-4)])
def test_single_block(oracle, blocks, name, g, eps):
    print("split", name, g, eps, flush=True)
    hb = blocks[name]
    run = D.StagedRun([hb])
    run.run(g, eps=eps)
    st = run.sync()
    out = run.fetch(0, volumes=True)
    s, npts = run.cells(0)
    ob = oracle.Block.from_host(hb)
    want = oracle.dense_single(ob, g, eps=eps)
    assert np.array_equal(s, want["status"])
    assert np.array_equal(npts, want["npts"])
    assert np.array_equal(_bits(out["density"]), _bits(want["density"]))
    vol = oracle.volumes(ob)
    assert np.array_equal(_bits(out["volumes"]), _bits(vol))
    assert np.array_equal(_bits(D.volumes(hb)), _bits(vol))
    if name == "uniform":
        assert st["cells_deferred"] >= 1   # stars beyond the tables


@pytest.mark.parametrize("counts", [(1, 200), (63, 130), (64, 65)])
@pytest.mark.parametrize("g", [11, 30])
def test_tile_edges(oracle, counts, g):
    print("split tiles", counts, g, flush=True)
    rng = np.random.default_rng(sum(counts))
    pts, bid, bounds = [], [], []
    for b, n in enumerate(counts):
        lo, hi = np.array([0.5 * b, 0, 0]), np.array([0.5 * (b + 1), 1, 1])
        pts.append((lo + rng.random((n, 3)) * (hi - lo)).astype(np.float32))
        bid.append(np.full(n, b))
        bounds.append((lo.astype(np.float32), hi.astype(np.float32)))
    blocks = ingest.decomposed_blocks(np.concatenate(pts), np.concatenate(bid), bounds, 0.5)
    res = D.dense(D.DENSE_TESS, 0, None, None, False, None, 1.0, 1e-4, (g, g, g), blocks,
                  want_cells=True)
    want = oracle.dense_multi([oracle.Block.from_host(b) for b in blocks], (g, g, g))
    for i in range(2):
        assert np.array_equal(res.cells[i][0], want["status"][i])
        assert np.array_equal(res.cells[i][1], want["npts"][i])
        assert np.array_equal(_bits(res.density[i]), _bits(want["density"][i])), i
