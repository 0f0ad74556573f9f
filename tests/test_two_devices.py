"""Host code on a stub of the HIP runtime, in a process of its own: the large-LDS kernels are prepared on each
device that runs them; a batch's first run of a step count allocates and copies once."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
INCLUDE = "/opt/rocm/include"

CHILD = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the real runtime
import numpy as np
from convstencil_amd import Layout, _lib
lib = _lib.load()
lib.cs_debug_variant_info.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                                      ctypes.c_char_p, ctypes.c_int32]
bad = []
for family in (2, 8, 10, 11, 12):
    for i in range(lib.cs_debug_variant_count(family)):
        info = (ctypes.c_int64 * 12)()
        lib.cs_debug_variant_info(family, i, info, None, 0)
        r = int(info[2])
        if family == 2 and info[1] != 4:
            continue
        L = Layout.with_halo([300, 1200], r)
        w = np.full((2 * r + 1, 2 * r + 1), 0.01)
        if info[3]:
            w[:r, :r] = w[:r, r + 1:] = w[r + 1:, :r] = w[r + 1:, r + 1:] = 0.0
        st = _lib.cs_stencil(2, r, w.ctypes.data_as(_lib.c_double_p))
        opt = _lib.cs_options()
        opt.tile_variant = int(info[0])
        Lc, fin = L.to_c(), ctypes.c_int32(-1)
        for dev in (0, 1):
            stub.hipSetDevice(dev)
            rc = lib.cs_run_2d_noalloc(ctypes.byref(Lc), ctypes.byref(st), ctypes.c_void_p(4096), ctypes.c_void_p(8192),
                                       2 * int(info[4]) + 1, ctypes.byref(opt), None, ctypes.byref(fin))
            if rc != 0:
                bad.append((int(info[0]), dev, rc))
print("launches", stub.stub_launches(), "refused", stub.stub_refused(), "bad", bad)
sys.exit(1 if bad or stub.stub_refused() or not stub.stub_launches() else 0)
"""


BATCH = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from convstencil_amd import Batch, Layout, dense_weights, shape_offsets
items = []
for shape, r, ny, nx in (("box2d1r", 1, 300, 400), ("box2d1r", 1, 200, 150), ("star2d3r", 3, 500, 300),
                         ("star2d3r", 3, 300, 200), ("box2d1r", 1, 20, 90)):
    offs = shape_offsets(shape)
    items.append((Layout.with_halo([ny, nx], r), r, dense_weights(2, r, offs, np.full(len(offs), 1.0 / len(offs)))))
with Batch(*zip(*items)) as b:
    for g, (L, r, w) in enumerate(items):
        b.upload(g, np.zeros(L.cells))
    before = stub.stub_mallocs(), stub.stub_copies()
    n0 = stub.stub_launches()
    b.run(500)
    mallocs, copies = stub.stub_mallocs() - before[0], stub.stub_copies() - before[1]
    launches = stub.stub_launches() - n0
    print("launches", launches, "allocations", mallocs, "copies", copies)
    # one buffer with every list of items, one copy into it, one of the grid table and one of the error word
    ok = launches > 200 and mallocs <= 1 and copies <= 3
print("allocations", stub.stub_mallocs(), "freed", stub.stub_frees())
sys.exit(0 if ok and stub.stub_mallocs() == stub.stub_frees() else 1)
"""

NEEDS = pytest.mark.skipif(not shutil.which("g++") or not os.path.isdir(INCLUDE), reason="needs g++ and the HIP headers")


def _run_on_stub(tmp_path, child):
    so = str(tmp_path / "hip_stub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", INCLUDE,
                    os.path.join(HERE, "hip_stub.cpp"), "-o", so], check=True, timeout=120)
    p = subprocess.run([sys.executable, "-c", child, so], cwd=os.path.dirname(HERE), capture_output=True, text=True,
                       timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr


@NEEDS
def test_kernels_are_prepared_on_every_device(tmp_path):
    _run_on_stub(tmp_path, CHILD)


@NEEDS
def test_a_batch_uploads_its_launch_lists_at_once(tmp_path):
    _run_on_stub(tmp_path, BATCH)
