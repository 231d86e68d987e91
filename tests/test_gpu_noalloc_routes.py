"""tess2_volumes_noalloc above 4096 cells (two cells a wave) and above 16384
(the geometry kernel), the caller's order as it is: volumes with the bits of
tess2_volumes, and a block with an index out of range refused with the output
as it was, by a mark its kernels see before they read the block."""
import ctypes as C

import numpy as np
import pytest

from tess2_amd import _native as N
from tess2_amd import host as D
from tess2_amd import ingest, synthetic

pytestmark = pytest.mark.gpu

E_ARG = -1      # TESS2_E_ARG


def _bits(a):
    a = np.ascontiguousarray(a, np.float32).ravel()
    return np.where(np.isnan(a), np.float32(np.nan), a).view(np.uint32)


@pytest.fixture
def put():
    """Device copies of arrays, through the runtime the library links."""
    N.lib()
    rt = C.CDLL("libamdhip64.so.7")
    bufs = []

    def copy(a):
        a = np.ascontiguousarray(a)
        p = C.c_void_p()
        assert rt.hipMalloc(C.byref(p), C.c_size_t(a.nbytes)) == 0
        bufs.append(p)
        assert rt.hipMemcpy(p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1) == 0
        return p.value

    def get(p, n):
        a = np.zeros(n, np.float32)
        assert rt.hipMemcpy(a.ctypes.data_as(C.c_void_p), C.c_void_p(p), C.c_size_t(a.nbytes),
                            2) == 0
        return a

    copy.get = get
    yield copy
    for p in bufs:
        rt.hipFree(p)


@pytest.mark.parametrize("n", [4096, 4097, 5000, 16383, 16384, 20000])
def test_good_and_refused(put, n):
    print("noalloc routes", n, flush=True)
    hb = ingest.periodic_block(synthetic.uniform(n, seed=n), 3.0 / n ** (1 / 3))
    want = _bits(D.volumes(hb))
    p, v = put(hb.particles), put(hb.vert_to_tet)
    t = put(hb.tets)
    out = put(np.full(n, -7.0, np.float32))
    ctx = N.Context(0)

    def call(tets, v2t):
        return N.lib().tess2_volumes_noalloc(ctx.h, p, hb.num_particles, n, tets, hb.num_tets, v2t,
                                             out)

    bad = []
    for col, x in ((2, hb.num_particles), (0, -1), (5, hb.num_tets), (7, -2)):
        a = hb.tets.copy()
        a[len(a) // 2, col] = x
        bad.append((put(a), v))
    a = hb.vert_to_tet.copy()
    a[-1] = hb.num_tets
    bad.append((t, put(a)))
    for tets, v2t in bad:
        assert call(tets, v2t) == E_ARG
        assert np.all(put.get(out, n) == np.float32(-7.0))
    assert call(t, v) == 0
    got = put.get(out, n)
    assert np.array_equal(_bits(got), want)
    # a refused call behind a good one leaves its volumes
    assert call(*bad[0]) == E_ARG
    assert np.array_equal(_bits(put.get(out, n)), want)
    assert call(t, v) == 0
    assert np.array_equal(_bits(put.get(out, n)), want)
