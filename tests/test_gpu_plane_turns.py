"""A scan whose planes are held for a few tiles at a time: turns behind the
first (their own list of large boxes, planes over the ones before), one block
and several, against one turn and the oracle."""
import numpy as np
import pytest

from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu


def _bits(a):
    a = np.ascontiguousarray(a, np.float32).ravel()
    return np.where(np.isnan(a), np.float32(np.nan), a).view(np.uint32)


def _one():
    # 16,500 cells (258 tiles); the sparse half has boxes beyond a tile's lines
    rng = np.random.default_rng(8)
    p = rng.random((16500, 3))
    p[:14000] *= 0.35
    p = np.unique(p.astype(np.float32), axis=0)
    rng.shuffle(p)
    return [ingest.make_block(p, len(p), (0, 0, 0), (1, 1, 1))]


def _several():
    p = synthetic.uniform(1500, seed=3)
    p[:900] *= np.float32(0.4)
    p = np.unique(p, axis=0)
    ids = (p[:, 0] >= 0.3).astype(int)
    bounds = [((0, 0, 0), (0.3, 1, 1)), ((0.3, 0, 0), (1, 1, 1))]
    return ingest.decomposed_blocks(p, ids, bounds, 0.3)


def _lattice(n):
    """n^3 nearly regular points, every cube of the lattice cut into six tets
    along its diagonal (base, base + e_a, base + e_a + e_b, opposite corner, for
    each order of the axes): a closed star for every inner point at once."""
    perms = [(0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)]
    stride = np.array([1, n, n * n])
    m = n - 1
    cube = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:, ::-1]
    base = cube @ stride
    cid = cube @ np.array([1, m, m * m])
    t = np.empty((len(cube), 6, 8), np.int32)
    for k, (a, b, c) in enumerate(perms):
        t[cid, k, 0] = base
        t[cid, k, 1] = base + stride[a]
        t[cid, k, 2] = base + stride[a] + stride[b]
        t[cid, k, 3] = base + stride.sum()

        def across(axis, step, perm):     # the tet of another cube, -1 outside
            ok = (cube[:, axis] + step >= 0) & (cube[:, axis] + step < m)
            return np.where(ok, 6 * (cid + step * m ** axis) + perms.index(perm), -1)

        t[cid, k, 4] = across(a, 1, (b, c, a))
        t[cid, k, 5] = 6 * cid + perms.index((b, a, c))
        t[cid, k, 6] = 6 * cid + perms.index((a, c, b))
        t[cid, k, 7] = across(c, -1, (c, a, b))
    t = t.reshape(-1, 8)
    v2t = np.full(n ** 3, -1, np.int32)
    for i in range(4):
        v2t[t[:, i]] = np.arange(len(t), dtype=np.int32)
    rng = np.random.default_rng(n)
    x = np.arange(n)
    p = np.stack(np.meshgrid(x, x, x, indexing="ij"), -1).reshape(-1, 3)[:, ::-1]
    p = ((p + 0.5 + 0.05 * rng.random(p.shape)) / n).astype(np.float32)
    return ingest.HostBlock(p, t, v2t, n ** 3, np.zeros(3, np.float32), np.ones(3, np.float32))


@pytest.mark.parametrize("make,most", [(_one, 100), (_one, 129), (_several, 1), (_several, 7)])
def test_turns(oracle, make, most):
    print("plane turns", make.__name__, most, flush=True)
    blocks = make()
    g = (96, 96, 96)
    run = D.StagedRun(blocks)
    run.set_option("plane_tiles", most)
    for _ in range(2):                   # the second on planes with contents
        run.run(g)
        st = run.sync()
    got = [run.fetch(b, volumes=True) for b in range(len(blocks))]
    cells = [run.cells(b) for b in range(len(blocks))]
    run.set_option("plane_tiles", 32768)
    run.run(g)
    st1 = run.sync()
    for b in range(len(blocks)):
        one = run.fetch(b, volumes=True)
        assert np.array_equal(_bits(got[b]["density"]), _bits(one["density"]))
        assert np.array_equal(_bits(got[b]["volumes"]), _bits(one["volumes"]))
        assert all(np.array_equal(x, y) for x, y in zip(cells[b], run.cells(b)))
    for k in ("cells_scan", "cells_cic", "points_deposited", "points_shared", "cells_deferred"):
        assert st[k] == st1[k]
    if len(blocks) == 1:
        want = oracle.dense_single(oracle.Block.from_host(blocks[0]), g)
        assert np.array_equal(_bits(got[0]["density"]), _bits(want["density"]))


def test_more_cells_than_one_turn_holds():
    """2,146,689 cells (33,543 tiles) in two turns: the two-cell kernel's bits."""
    hb = _lattice(129)
    print("plane turns", hb.num_orig, flush=True)
    run = D.StagedRun([hb])
    g = (150, 150, 150)
    run.run(g)
    a = run.sync()
    da, (sa, na) = run.fetch(0, volumes=True), run.cells(0)
    run.set_option("cell_kernel", 1)
    run.run(g)
    b = run.sync()
    db, (sb, nb) = run.fetch(0, volumes=True), run.cells(0)
    assert a["cells_scan"] + a["cells_cic"] > 2_000_000
    assert all(a[k] == b[k] for k in ("cells_scan", "cells_cic", "points_deposited"))
    assert np.array_equal(sa, sb) and np.array_equal(na, nb)
    assert np.array_equal(_bits(da["density"]), _bits(db["density"]))
    assert np.array_equal(_bits(da["volumes"]), _bits(db["volumes"]))
