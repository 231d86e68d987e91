"""Staging where its sort changes the size of its tiles (65,536 and 131,072
particles) and with ghosts between the originals: volumes in the caller's
order equal the oracle's bit for bit."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu


def _bits(a):
    a = np.ascontiguousarray(a, np.float32).ravel()
    return np.where(np.isnan(a), np.float32(np.nan), a).view(np.uint32)


@pytest.mark.parametrize("n,norig", [(65536, 65536), (65537, 40000), (131073, 131073)])
def test_layout_tiles(oracle, n, norig):
    print("stage tiles", n, norig, flush=True)
    p = synthetic.uniform(n, seed=n)
    hb = ingest.make_block(p, norig, (0, 0, 0), (1, 1, 1))
    want_cc = oracle.circumcenters(hb.tets, hb.particles)
    want = oracle.volumes(oracle.Block.from_host(hb), want_cc)
    assert np.array_equal(_bits(D.volumes(hb)), _bits(want))
    run = D.StagedRun([hb])
    run.run((16, 16, 16))
    run.sync()
    out = run.fetch(0, volumes=True, circumcenters=True)
    assert np.array_equal(_bits(out["circumcenters"]), _bits(want_cc))
    assert np.array_equal(_bits(out["volumes"]), _bits(want))
