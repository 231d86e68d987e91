"""The exact assignment on boxes far from zero, where a coordinate's ulp is a
good part of a bucket: owners equal the FP64 oracle's in both precisions."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [D.MIXED, D.FP64])
@pytest.mark.parametrize("off", [1000.0, -20000.0])
@pytest.mark.parametrize("extent", [(1.0, 1.0, 1.0), (1.0, 1.0, 0.05)])
def test_offset_box(oracle, off, extent, prec):
    print("owner offset", off, extent, prec, flush=True)
    rng = np.random.default_rng(int(abs(off)))
    ext = np.array(extent)
    p = np.unique((off + rng.random((3000, 3)) * ext).astype(np.float32), axis=0)
    rng.shuffle(p)
    lo = np.full(3, off, np.float32)
    # tessellated about the origin (the differences are exact), then put in place
    hb = ingest.make_block((p - lo).astype(np.float32), len(p), (0, 0, 0), extent)
    hb.particles, hb.bounds_min, hb.bounds_max = p, lo, (lo + ext).astype(np.float32)
    g = (31, 31, 7)
    run = D.StagedRun([hb])
    run.run(g, assignment=D.EXACT_VORONOI, precision=prec, want_volumes=False)
    run.sync()
    want = oracle.exact_dense(oracle.Block.from_host(hb), g)
    assert np.array_equal(run.owner(0), want["owner"])
