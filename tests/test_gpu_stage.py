"""Staging on the device (range checks, bounding box, Morton order of cells
and tets) where its tiles, scans and digit passes have their edges: volumes,
circumcenters (in the caller's tet numbering) and densities are the oracle's
bit for bit, and out-of-range indices are refused by name."""
import sys

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


def _block(name):
    if name == "one_tet":
        p = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32)
        t = np.array([[0, 1, 2, 3, -1, -1, -1, -1]], np.int32)
        return ingest.HostBlock(p, t, np.zeros(4, np.int32), 4, np.zeros(3, np.float32),
                                np.ones(3, np.float32))
    if name == "no_tets":
        p = synthetic.uniform(65, seed=2)
        return ingest.HostBlock(p, np.zeros((0, 8), np.int32), np.full(65, -1, np.int32), 65,
                                np.zeros(3, np.float32), np.ones(3, np.float32))
    if name == "one_cluster":
        # nearly all particles share one Morton code: ties stay in id order
        p = synthetic.uniform(1500, seed=4)
        p[:1400] = np.float32(0.5) + p[:1400] * np.float32(2e-4)
        return ingest.make_block(p, 1500, (0, 0, 0), (1, 1, 1))
    n = int(name)
    return ingest.periodic_block(synthetic.uniform(n, seed=n), 4.0 / n ** (1 / 3))


# 1024-particle order tiles, 4096-pair sort tiles, and more than 64 sort tiles
# of tets (the digit scan's second level), where the particles end in a tile
@pytest.mark.parametrize("name", ["one_tet", "no_tets", "one_cluster", "130", "1024", "1025",
                                  "21001"])
def test_staged_order(oracle, name):
    print("staging", name, flush=True)
    sys.stdout.flush()
    hb = _block(name)
    ob = oracle.Block.from_host(hb)
    want_cc = oracle.circumcenters(hb.tets, hb.particles)
    want_vol = oracle.volumes(ob, want_cc)
    g = (24, 24, 24)
    run = D.StagedRun([hb])
    run.run(g)
    run.sync()
    out = run.fetch(0, volumes=True, circumcenters=True)
    assert np.array_equal(_bits(out["circumcenters"]), _bits(want_cc))
    assert np.array_equal(_bits(out["volumes"]), _bits(want_vol))
    assert np.array_equal(_bits(out["density"]), _bits(oracle.dense_single(ob, g)["density"]))
    # the one-call forms: the caller's order, and buffers given back in between
    for _ in range(2):
        assert np.array_equal(_bits(D.fill_circumcenters(hb.tets, hb.particles)), _bits(want_cc))
        assert np.array_equal(_bits(D.volumes(hb)), _bits(want_vol))


def test_cic_then_scan_on_one_context(oracle):
    """A CIC call stages no Morton order; a later scan of the same staged
    block makes it."""
    hb = _block("1025")
    g = (24, 24, 24)
    ctx = D.N.Context(0)
    D.dense(D.DENSE_CIC, 0, None, None, False, None, 1.0, 1e-4, g, [hb], ctx=ctx)
    r = D.StagedRun.__new__(D.StagedRun)
    r.ctx, r.blocks = ctx, [hb]
    r.run(g)
    r.sync()
    want = oracle.dense_single(oracle.Block.from_host(hb), g)["density"]
    assert np.array_equal(_bits(r.fetch(0)["density"]), _bits(want))


def test_refused_input_keeps_the_staged_block(oracle):
    hb = _block("130")
    run = D.StagedRun([hb])
    bad = _block("130")
    bad.tets = bad.tets.copy()
    bad.tets[7, 6] = len(bad.tets)
    with pytest.raises(D.Tess2Error, match="tet 7 neighbour"):
        D.volumes(bad, ctx=run.ctx)
    bad = _block("130")
    bad.vert_to_tet = bad.vert_to_tet.copy()
    bad.vert_to_tet[129] = -2
    with pytest.raises(D.Tess2Error, match=r"vert_to_tet\[129\]"):
        D.volumes(bad, ctx=run.ctx)
    g = (24, 24, 24)
    run.run(g)
    run.sync()
    want = oracle.dense_single(oracle.Block.from_host(hb), g)["density"]
    assert np.array_equal(_bits(run.fetch(0)["density"]), _bits(want))
