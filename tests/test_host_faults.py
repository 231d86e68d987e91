"""The library's host paths on a HIP runtime without a GPU (fake_hip.py): what
a failed copy, allocation or thread leaves behind, what a run keeps from the run
before, and which kernels a choice reaches."""
import ctypes as C
import shutil

import numpy as np
import pytest

from tess2_amd import _native as N
from tess2_amd import build as B
from tess2_amd import host as D
from tess2_amd import ingest
from tests import fake_hip as F

E_HIP, E_NOMEM = -2, -4
MIB = 1 << 20


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    try:
        B.hipcc()
    except RuntimeError:
        pytest.skip("hipcc missing")
    if shutil.which("g++") is None:
        pytest.skip("g++ missing")
    return F.load(F.build(str(tmp_path_factory.mktemp("fake"))))


@pytest.fixture
def fake(lib, monkeypatch):
    monkeypatch.setattr(N, "_lib", lib)
    # a context collected later would be closed by another library
    monkeypatch.setattr(N.Context, "__del__", lambda self: None)
    lib.fake_reset()
    yield lib
    lib.fake_reset()


def _block(n, seed=1, gid=0):
    """n particles without ghosts or neighbours, enough for the host code."""
    rng = np.random.default_rng(seed)
    p = rng.random((n, 3), dtype=np.float32)
    t = np.full((n, 8), -1, np.int32)
    t[:, :4] = np.arange(4)
    hb = ingest.HostBlock(p, t, np.zeros(n, np.int32), n, np.zeros(3, np.float32),
                          np.ones(3, np.float32))
    hb.gid = gid
    return hb


def _stage(ctx, blocks):
    cs = (N.Block * len(blocks))()
    keep = []
    for i, hb in enumerate(blocks):
        cs[i], k = N.make_block(hb)
        keep.append(k)
    return N.lib().tess2_stage(ctx.h, cs, len(blocks)), keep


# ---- failed copies ----------------------------------------------------------
@pytest.mark.parametrize("nth", [1, 2, 3])
def test_failed_upload_leaves_no_copy_of_the_callers_arrays(fake, nth):
    """The caller may free its arrays when an error is returned."""
    ctx = N.Context(0)
    fake.fake_fail_copy(nth)
    r, _ = _stage(ctx, [_block(1000)])
    assert r == E_HIP
    assert fake.fake_pending() == 0
    fake.fake_fail_copy(-1)
    assert _stage(ctx, [_block(1000)])[0] == 0


def test_failed_ghost_test_leaves_no_copy_of_the_boxes(fake):
    hb = _block(1000)
    boxes = np.zeros((3, 6), np.float32)
    ctx = N.Context(0)
    D.ghost_sends(hb, boxes, ctx=ctx)
    n = fake.fake_copies()
    fake.fake_fail_copy(n - 1)          # the last copy of a call: the result
    with pytest.raises(N.Tess2Error):
        D.ghost_sends(hb, boxes, ctx=ctx)
    assert fake.fake_pending() == 0
    D.ghost_sends(hb, boxes, ctx=ctx)


def test_no_memory_for_copy_threads(fake):
    """A large copy goes on with the threads that started."""
    run = D.StagedRun([_block(500)])
    g = (256, 256, 128)
    run.run(g)
    run.sync()
    out = np.ones(g[0] * g[1] * g[2], np.float32)
    assert N.lib().tess2_fetch(run.ctx.h, 0, out.ctypes.data, None, None) == 0
    out[:] = 1.0
    for n in range(4):      # the threads' own states
        fake.fake_fail_new(n)
        r = N.lib().tess2_fetch(run.ctx.h, 0, out.ctypes.data, None, None)
        fake.fake_fail_new(-1)
        assert r == 0 and not out.any()
        out[:] = 1.0


# ---- pinned arrays ----------------------------------------------------------
def test_pinned_arrays_are_copied_directly(fake):
    """An array the device reaches by itself needs no slots in between."""
    n = (20 << 20) // 32                       # tets above the least upload in slots
    hb = _block(n)
    t = fake.fake_pinned(hb.tets.nbytes)
    C.memmove(t, hb.tets.ctypes.data, hb.tets.nbytes)
    b, keep = N.make_block(hb)
    b.tets = t
    ctx = N.Context(0)
    assert N.lib().tess2_stage(ctx.h, C.byref(b), 1) == 0
    direct = fake.fake_copies()
    assert direct == 4                         # three arrays up, the check's record down

    run = D.StagedRun([_block(500)])
    g = (256, 256, 128)
    run.run(g)
    run.sync()
    d = fake.fake_pinned(4 * g[0] * g[1] * g[2])
    before = fake.fake_copies()
    assert N.lib().tess2_fetch(run.ctx.h, 0, d, None, None) == 0
    assert fake.fake_copies() == before + 1


# ---- failed allocations -----------------------------------------------------
@pytest.mark.parametrize("mib", [0, 10, 40, 75, 140, 200, 210])
def test_run_after_a_run_without_memory(fake, mib):
    """A run on a larger grid finds no memory part of the way; the smaller grid
    then runs on buffers that are all there."""
    run = D.StagedRun([_block(2000)])
    kw = dict(assignment=D.EXACT_VORONOI, want_volumes=False)
    run.run((33, 33, 33), **kw)
    run.sync()
    fake.fake_limit(mib * MIB)
    with pytest.raises(N.Tess2Error, match="out of device memory"):
        run.run((200, 200, 200), **kw)
    fake.fake_limit(2 ** 64 - 1)
    run.run((33, 33, 33), **kw)
    run.sync()
    run.run((20, 20, 20))
    run.sync()
    assert fake.fake_bad_launches() == 0


def test_run_after_a_staging_without_memory(fake):
    """Whatever allocation of a staging fails, the next run has all its buffers
    (the blocks staged before) or is refused."""
    blocks = [_block(300, 1, 0), _block(200, 2, 1)]
    ctx = N.Context(0)
    g = N.i3((9, 9, 9))

    def run():
        r = N.lib().tess2_run(ctx.h, 0, 0, N.f3(None), N.f3(None), 0, N.f3((0, 0, 1)), 1.0, 1e-4,
                              g, 0, 0, 0)
        return r or N.lib().tess2_sync(ctx.h, None)

    refused = staged = 0
    for kib in range(0, 1500, 8):
        fake.fake_limit(kib << 10)
        r, _ = _stage(ctx, blocks)
        fake.fake_limit(2 ** 64 - 1)
        assert r in (0, E_NOMEM)
        staged += r == 0
        if run():
            assert b"no staged blocks" in N.lib().tess2_last_error(ctx.h)
            refused += 1
        assert fake.fake_bad_launches() == 0
        N.lib().tess2_destroy(ctx.h)        # the next without buffers of this one
        ctx = N.Context(0)
    assert refused and staged


def _runs(run, g=(9, 9, 9)):
    run.run(g, want_volumes=False)
    run.sync()


def test_planes_without_memory(fake):
    """The planes between the geometry and the scan kernel (4097 tiles of 42 KB)
    are held in fewer tiles at a time where memory is short, and a run that finds
    none takes the one-pass kernel, as it did without planes."""
    n = 64 * 4096 + 1
    hb = _block(n)
    turns = {}
    for mib in (400, 100, 60, 30, 0):
        run = D.StagedRun([hb])
        run.set_option("cell_kernel", 1)        # all other buffers
        _runs(run)
        run.set_option("cell_kernel", -1)
        fake.fake_limit(mib * MIB)
        before = [fake.fake_launches(k) for k in (F.K_GEOM, F.K_SCAN, F.K_MC)]
        _runs(run)
        _runs(run)
        fake.fake_limit(2 ** 64 - 1)
        turns[mib] = [fake.fake_launches(k) - b
                      for k, b in zip((F.K_GEOM, F.K_SCAN, F.K_MC), before)]
        assert fake.fake_bad_launches() == 0
        # the next staging has its planes again
        assert _stage(run.ctx, [hb])[0] == 0
        before = fake.fake_launches(F.K_GEOM)
        _runs(run)
        assert fake.fake_launches(F.K_GEOM) == before + 1
        run.ctx.close()
    assert turns == {400: [2, 2, 0], 100: [4, 4, 0], 60: [8, 8, 0], 30: [0, 0, 2], 0: [0, 0, 2]}


def test_plane_turns_are_equal(fake):
    run = D.StagedRun([_block(64 * 1000 + 5)])      # 1001 tiles
    for most, turns in ((32768, 1), (1001, 1), (1000, 2), (400, 3), (1, 1001)):
        run.set_option("plane_tiles", most)
        assert run.get_option("plane_tiles") == most
        before = fake.fake_launches(F.K_GEOM)
        _runs(run)
        assert fake.fake_launches(F.K_GEOM) - before == turns
        assert fake.fake_bad_launches() == 0
    for bad in (0, 32769):
        with pytest.raises(N.Tess2Error):
            run.set_option("plane_tiles", bad)


def test_cic_list_without_memory(fake):
    """A CIC run's list holds eight contributions a cell where there is memory,
    and starts as small as a scan's where there is not."""
    hb = _block(400000)
    for mib in (4000, 60):
        run = D.StagedRun([hb])
        fake.fake_limit(mib * MIB)
        run.run((9, 9, 9), alg=D.DENSE_CIC)
        run.sync()
        fake.fake_limit(2 ** 64 - 1)
        assert fake.fake_bad_launches() == 0
        run.ctx.close()


# ---- what a run keeps -------------------------------------------------------
@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("nb", [1, 2])
def test_fetching_leaves_the_next_run_its_descriptors(fake, graph, nb):
    """A steady state of run and fetch uploads nothing and records no graph
    again, whatever is fetched."""
    run = D.StagedRun([_block(500, k, k) for k in range(nb)])
    run.set_option("graph", graph)
    _runs(run)
    _runs(run)
    before = fake.fake_copies()
    _runs(run)
    steady, graphs = fake.fake_copies() - before, fake.fake_graphs()
    for _ in range(3):
        run.fetch(0, circumcenters=True)
        run.cells(0)
        before = fake.fake_copies()
        _runs(run)
        assert fake.fake_copies() - before == steady
    assert fake.fake_graphs() == graphs


# ---- the tuned cell kernel --------------------------------------------------
KERNELS = {3: F.K_REF_BATCHED, 1: F.K_MC_BATCHED, 4: F.K_MC_ITEMS, -1: F.K_GEOM}


def _used(fake, run, **kw):
    before = {k: fake.fake_launches(k) for k in range(8)}
    run.run((9, 9, 9), **kw)
    run.sync()
    return {k for k in range(1, 8) if fake.fake_launches(k) > before[k]}


@pytest.mark.parametrize("best", [3, 1, 4, -1])
def test_tuned_kernel_is_for_several_blocks(fake, best):
    """What tess2_autotune chooses for several blocks is neither the choice for
    a single block staged later nor the end of the choice."""
    for k in KERNELS.values():
        fake.fake_cost(k, 1.0)
    fake.fake_cost(KERNELS[best], 0.01)
    run = D.StagedRun([_block(300, 1, 0), _block(200, 2, 1)])
    _runs(run)
    run.autotune(reps=1)
    assert run.get_option("cell_kernel") == best
    assert KERNELS[best] in _used(fake, run, want_volumes=False)
    # one block: the geometry and scan kernels, and the automatic volumes
    big, few = _block(20000), _block(300)
    assert _stage(run.ctx, [big])[0] == 0
    run.blocks = [big]
    assert _used(fake, run, want_volumes=False) == {F.K_GEOM, F.K_SCAN}
    D.volumes(few, ctx=run.ctx)
    assert _stage(run.ctx, [few])[0] == 0
    run.blocks = [few]
    assert _used(fake, run, want_volumes=False) == {F.K_MC}
    # another set of blocks is tuned over all kernels again
    blocks = [_block(100, 1, 0), _block(900, 2, 1)]
    assert _stage(run.ctx, blocks)[0] == 0
    run.blocks = blocks
    _runs(run)
    for now, k in KERNELS.items():
        fake.fake_cost(k, 0.01 if now == 4 else 1.0)
    run.autotune(reps=1)
    assert run.get_option("cell_kernel") == 4


def test_asked_kernel_stays(fake):
    run = D.StagedRun([_block(300, 1, 0), _block(200, 2, 1)])
    run.set_option("cell_kernel", 1)
    _runs(run)
    run.autotune(reps=1)
    assert run.get_option("cell_kernel") == 1
    few = _block(20000)
    assert _stage(run.ctx, [few])[0] == 0
    run.blocks = [few]
    assert _used(fake, run, want_volumes=False) == {F.K_MC}


def test_runs_without_cell_kernels_choose_none(fake):
    """The time of a CIC run says nothing about the cell kernels."""
    run = D.StagedRun([_block(300, 1, 0), _block(200, 2, 1)])
    fake.fake_cost(F.K_OTHER, 1.0)
    fake.fake_drift(0.999)              # every candidate looks faster than the one before
    for kw in (dict(alg=D.DENSE_CIC), dict(assignment=D.EXACT_VORONOI, want_volumes=False)):
        run.run((9, 9, 9), **kw)
        run.sync()
        before = sum(fake.fake_launches(k) for k in range(1, 8))
        run.autotune(reps=1)
        assert run.get_option("cell_kernel") == -1
        assert sum(fake.fake_launches(k) for k in range(1, 8)) == before


def test_few_grid_points_take_the_one_pass_kernel(fake):
    one, two = D.StagedRun([_block(20000)]), D.StagedRun([_block(300, 1, 0), _block(200, 2, 1)])
    for run, split in ((one, False), (two, True)):
        for g in ((3, 3, 3), (4, 4, 4), (2, 2, 16)):
            before = fake.fake_launches(F.K_SCAN)
            _runs(run, g)
            assert (fake.fake_launches(F.K_SCAN) > before) == (split or g != (3, 3, 3))


def test_small_results_come_in_one_waiting_copy(fake):
    """An asynchronous copy of up to 16 KB to pageable memory and a wait behind
    it take the runtime twice as long as a copy that waits."""
    run = D.StagedRun([_block(500)])
    _runs(run)
    before = fake.fake_copies()
    run.cells(0)
    run.fetch(0, volumes=False)
    run.fetch(0, ngrid=False, circumcenters=True)
    assert fake.fake_copies() == before + 4
    assert fake.fake_async_downloads() == 0
