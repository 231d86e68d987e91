"""The tile search of the exact assignment where its shells, rows and boxes
have their edges: grid tiles of one point, tiles that span many buckets,
points far from every particle and outside the particles' box, a bucket that
holds nearly all particles, and exact ties between shells.  Owners equal the
FP64 oracle's in both precisions."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu


def _block(name):
    rng = np.random.default_rng(77)
    if name == "corner":      # far points: many empty shells, one full bucket
        p = np.concatenate([rng.random((300, 3)) * 0.01 + 0.02,
                            [[0.9, 0.1, 0.2], [0.2, 0.95, 0.1], [0.1, 0.2, 0.9]]])
    elif name == "five":      # fewer buckets than a tile's shell
        p = rng.random((5, 3)) * 0.2 + 0.4
    elif name == "slab":      # one bucket thick along z
        p = rng.random((400, 3)) * [1.0, 1.0, 0.004] + [0, 0, 0.5]
    else:                     # ties: points midway between sites of different shells
        return ingest.periodic_block(synthetic.jittered_lattice(4, 0.0, seed=1), 3.0 / 4)
    return ingest.make_block(p.astype(np.float32), len(p), (0, 0, 0), (1, 1, 1))


@pytest.mark.parametrize("prec", [D.MIXED, D.FP64])
@pytest.mark.parametrize("name", ["corner", "five", "slab", "ties"])
@pytest.mark.parametrize("g", [(5, 5, 5), (9, 9, 9), (34, 21, 18)])
def test_owner(oracle, name, g, prec):
    print("owner tiles", name, g, prec, flush=True)
    hb = _block(name)
    run = D.StagedRun([hb])
    run.run(g, assignment=D.EXACT_VORONOI, precision=prec, want_volumes=False)
    run.sync()
    want = oracle.exact_dense(oracle.Block.from_host(hb), g)
    assert np.array_equal(run.owner(0), want["owner"])
    s, n = run.cells(0)
    assert np.array_equal(s, want["status"]) and np.array_equal(n, want["npts"])
