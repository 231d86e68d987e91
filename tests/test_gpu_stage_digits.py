"""Staging of more particles than one workgroup scans the sort's digit counts
of (262,144 in 64 tiles), so that the counts take the scan over tiles: originals
and ghosts, a cluster whose particles share Morton codes, and unconnected tets.
Circumcenters come back in the caller's numbering with the oracle's bits, which
takes a whole renumbering, and every original cell is visited."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest

pytestmark = pytest.mark.gpu

INCOMPLETE = 2      # a cell at a face without a neighbour


def _bits(a):
    a = np.ascontiguousarray(a, np.float32).ravel()
    return np.where(np.isnan(a), np.float32(np.nan), a).view(np.uint32)


@pytest.mark.parametrize("n,norig", [(262144, 262144), (262145, 200003), (600011, 300007)])
def test_many_digit_tiles(oracle, n, norig):
    print("stage digits", n, norig, flush=True)
    rng = np.random.default_rng(n)
    p = rng.random((n, 3), dtype=np.float32)
    p[::3] = np.float32(0.25) + p[::3] * np.float32(1e-3)
    t = np.full((n // 4, 8), -1, np.int32)
    t[:, :4] = rng.permutation(n)[: n // 4 * 4].reshape(-1, 4)
    hb = ingest.HostBlock(p, t, ingest.vert_to_tet(t, n), norig, np.zeros(3, np.float32),
                          np.ones(3, np.float32))
    run = D.StagedRun([hb])
    run.run((8, 8, 8), want_volumes=False)
    st = run.sync()
    assert st["cells_incomplete"] == norig
    s, _ = run.cells(0)
    assert np.all(s == INCOMPLETE)
    got = run.fetch(0, circumcenters=True)["circumcenters"]
    want = oracle.circumcenters(t, p)
    assert np.array_equal(_bits(got), _bits(want))
