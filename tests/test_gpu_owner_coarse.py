"""The exact assignment on grids coarser than the particles, where a wave
searches for 8 points or one, and on grids of unlike steps, whose tiles are no
cubes: owners, statuses and counts equal the FP64 oracle's in both precisions,
one block and several, with exact ties."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu


def _block(name):
    if name == "ties":
        return ingest.periodic_block(synthetic.jittered_lattice(8, 0.0, seed=1), 3.0 / 8)
    p = synthetic.uniform(3000, seed=12)
    if name == "clump":      # one bucket holds a third of the particles
        p[:1000] = np.float32(0.6) + p[:1000] * np.float32(0.01)
        p = np.unique(p, axis=0)
        np.random.default_rng(3).shuffle(p)
    return ingest.periodic_block(p, 4.0 / 3000 ** (1 / 3))


@pytest.mark.parametrize("prec", [D.MIXED, D.FP64])
@pytest.mark.parametrize("name", ["uniform", "clump", "ties"])
@pytest.mark.parametrize("g", [(2, 2, 2), (3, 3, 3), (7, 7, 7), (13, 13, 13), (19, 20, 21),
                               (33, 33, 33), (40, 40, 4), (3, 40, 40), (101, 9, 10), (2, 70, 2)])
def test_owner(oracle, name, g, prec):
    print("owner coarse", name, g, prec, flush=True)
    hb = _block(name)
    run = D.StagedRun([hb])
    run.run(g, assignment=D.EXACT_VORONOI, precision=prec, want_volumes=False)
    run.sync()
    want = oracle.exact_dense(oracle.Block.from_host(hb), g)
    assert np.array_equal(run.owner(0), want["owner"])
    s, n = run.cells(0)
    assert np.array_equal(s, want["status"]) and np.array_equal(n, want["npts"])


@pytest.mark.parametrize("g", [(5, 5, 5), (21, 7, 30)])
def test_several_blocks(oracle, g):
    """The owner of a grid point on several blocks is that of the whole set."""
    print("owner coarse blocks", g, flush=True)
    p = synthetic.uniform(4000, seed=5)
    ids = (p[:, 0] >= 0.45).astype(int)
    bounds = [((0, 0, 0), (0.45, 1, 1)), ((0.45, 0, 0), (1, 1, 1))]
    blocks = ingest.decomposed_blocks(p, ids, bounds, 0.35)
    run = D.StagedRun(blocks)
    run.run(g, assignment=D.EXACT_VORONOI, want_volumes=False)
    run.sync()
    home = np.concatenate([np.flatnonzero(ids == b) for b in range(2)])
    first = np.array([0, int((ids == 0).sum())])
    one = D.StagedRun([ingest.make_block(p, len(p), (0, 0, 0), (1, 1, 1))])
    one.run(g, assignment=D.EXACT_VORONOI, want_volumes=False)
    one.sync()
    want = one.owner(0).reshape(g[::-1])
    x = np.linspace(0.0, 1.0, g[0])
    at = 0
    for b in range(2):
        o = run.owner(b)
        o = o.reshape(g[2], g[1], -1)
        mine = o >= 0
        got = home[first[o[mine] >> 23] + (o[mine] & 0x7FFFFF)]
        cols = np.arange(at, at + o.shape[2]) if b == 0 else np.arange(g[0] - o.shape[2], g[0])
        assert np.array_equal(got, want[:, :, cols][mine])
        assert mine.sum() > 0 and x.size == g[0]
