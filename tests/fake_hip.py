"""The library's host code on the CPU: api.hip and transfer.hip compiled for
the host only and linked with a HIP runtime whose device memory is host memory,
whose kernels do nothing and whose failures and launch costs the test sets
(fake_hip.cpp)."""
import ctypes as C
import os
import subprocess

from tess2_amd import _native as N
from tess2_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))

CONTROL = {
    "fake_reset": (None, []),
    "fake_limit": (None, [C.c_size_t]),          # hipMalloc fails beyond so many bytes more
    "fake_fail_copy": (None, [C.c_long]),        # copies until one fails
    "fake_fail_new": (None, [C.c_long]),         # allocations until operator new throws
    "fake_cost": (None, [C.c_int, C.c_double]),  # ms per launch of a kind
    "fake_drift": (None, [C.c_double]),          # cost of a launch in terms of the one before
    "fake_pending": (C.c_long, []),              # uploads from pageable memory not waited for
    "fake_launches": (C.c_long, [C.c_int]),
    "fake_copies": (C.c_long, []),
    "fake_pinned_copies": (C.c_long, []),
    "fake_graphs": (C.c_long, []),
    "fake_mallocs": (C.c_long, []),
    "fake_async_downloads": (C.c_long, []),      # to pageable memory
    "fake_bad_launches": (C.c_long, []),         # with a buffer missing or too small
    "fake_pinned": (C.c_void_p, [C.c_size_t]),
}
(K_OTHER, K_GEOM, K_SCAN, K_REF_BATCHED, K_MC_BATCHED, K_MC_ITEMS, K_REF, K_MC) = range(8)


def build(outdir):
    cc, objs = B.hipcc(), []
    for src in (os.path.join(B.CSRC, "api.hip"), os.path.join(B.CSRC, "transfer.hip"),
                os.path.join(HERE, "fake_hip.cpp")):
        obj = os.path.join(outdir, os.path.basename(src) + ".o")
        subprocess.check_call([cc, "--offload-host-only", "-x", "hip", "-O1", "-std=c++17", "-fPIC",
                               "-ffp-contract=off", "-Wno-unused-function", "-c", src, "-o", obj])
        objs.append(obj)
    for s in B.HOST_SOURCES:
        obj = os.path.join(outdir, s + ".o")
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-c", os.path.join(B.CSRC, s),
                               "-o", obj])
        objs.append(obj)
    # the device code that a host-only object refers to
    names = subprocess.check_output(["nm", "-u"] + objs, text=True).split()
    stub = os.path.join(outdir, "fatbin.cpp")
    with open(stub, "w") as f:
        for n in sorted({n for n in names if n.startswith("__hip_fatbin")}):
            f.write(f'extern "C" {{ char {n}[16]; }}\n')
    out = os.path.join(outdir, "libtess2_fake.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-Wl,-z,defs", "-o", out]
                          + objs + [stub, "-lpthread"])
    return out


def load(path):
    lib = C.CDLL(path)
    for name, (res, args) in {**N.SIGNATURES, **CONTROL}.items():
        f = getattr(lib, name)
        f.restype, f.argtypes = res, args
    return lib
