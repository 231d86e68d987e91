"""Large copies of two contexts at once: one takes the pinned slots, the other
goes the plain way, and both arrive whole; arrays that are pinned already."""
import ctypes as C
import threading

import numpy as np
import pytest

from tess2_amd import _native as N
from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu

G = (161, 160, 159)      # 16.4 MB


def _bits(a):
    return np.ascontiguousarray(a, np.float32).ravel().view(np.uint32)


def test_two_contexts_at_once(oracle):
    print("copies of two contexts", flush=True)
    blocks = [ingest.periodic_block(synthetic.uniform(3000, seed=s), 4.0 / 3000 ** (1 / 3))
              for s in (1, 2)]
    want = [_bits(oracle.dense_single(oracle.Block.from_host(b), G)["density"]) for b in blocks]
    # tets of 17 MB: uploads in slots
    n = 530000
    t = np.full((n, 8), -1, np.int32)
    t[:, :4] = np.arange(4)
    wide = ingest.HostBlock(blocks[0].particles, t, np.zeros(blocks[0].num_particles, np.int32),
                            0, np.zeros(3, np.float32), np.ones(3, np.float32))
    cc = D.fill_circumcenters(t, blocks[0].particles)[0]
    bad = []

    def work(k):
        try:
            run = D.StagedRun([blocks[k]])
            run.run(G, want_volumes=False)
            run.sync()
            for _ in range(8):
                if not np.array_equal(_bits(run.fetch(0)["density"]), want[k]):
                    bad.append(("density", k))
            for _ in range(3):
                c = D.fill_circumcenters(wide.tets, wide.particles, ctx=run.ctx)
                if not np.array_equal(_bits(c), _bits(np.broadcast_to(cc, c.shape))):
                    bad.append(("circumcenters", k))
        except Exception as e:   # a thread's own would be lost
            bad.append(e)

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for x in th:
        x.start()
    for x in th:
        x.join()
    assert not bad


def test_pinned_arrays():
    print("pinned arrays", flush=True)
    hb = ingest.periodic_block(synthetic.uniform(2000, seed=3), 4.0 / 2000 ** (1 / 3))
    run = D.StagedRun([hb])
    run.run(G, want_volumes=False)
    run.sync()
    want = run.fetch(0)["density"]
    rt = C.CDLL("libamdhip64.so.7")
    p = C.c_void_p()
    assert rt.hipHostMalloc(C.byref(p), C.c_size_t(want.nbytes), 0) == 0
    try:
        got = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), want.shape)
        got[:] = -1.0
        assert N.lib().tess2_fetch(run.ctx.h, 0, got.ctypes.data, None, None) == 0
        assert np.array_equal(_bits(got), _bits(want))
        del got
    finally:
        rt.hipHostFree(p)
