"""The register-tile 2-D FP64 kernels (k2d_block.hip) against the CPU oracle: every depth, at the
tile's own size, one cell more, an odd number of tiles, with zero and with alternating halos."""
import ctypes

import numpy as np
import pytest

from convstencil_amd import Plan, Layout, shape_offsets, dense_weights, _lib
from oracle import oracle
from refimpl import rel_errors

pytestmark = pytest.mark.gpu


def _variants():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    lib.cs_debug_variant_info.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                                          ctypes.c_char_p, ctypes.c_int32]
    out = []
    for i in range(lib.cs_debug_variant_count(12)):
        info = (ctypes.c_int64 * 12)()
        name = ctypes.create_string_buffer(128)
        lib.cs_debug_variant_info(12, i, info, name, 128)
        out.append((int(info[0]), int(info[2]), "star" if info[3] else "box", int(info[4]), int(info[5]), int(info[6]),
                    name.value.decode()))
    return out


VARIANTS = _variants()


@pytest.mark.parametrize("vid,r,kind,kf,by,bx,name", VARIANTS, ids=[v[6] for v in VARIANTS])
def test_every_block_variant(gpu, vid, r, kind, kf, by, bx, name):
    print(f"case {name}", flush=True)
    offs = shape_offsets(f"{kind}2d{r}r")
    w = oracle.fill_weights(len(offs), vid)
    for k, (ny, nx, halo) in enumerate([(by, bx, 0), (by + 1, bx + 1, 1), (2 * by + 5, 2 * bx - 3, 0),
                                        (by, 2 * bx + 7, 1)]):
        L = Layout.with_halo([ny, nx], r + (k & 1), k)
        x = np.random.default_rng(vid + k).uniform(-1, 1, L.cells) if halo else oracle.fill_data(L, vid + k)
        for steps in (kf, 2 * kf + 1):
            with Plan(L, r, dense_weights(2, r, offs, w), variant=vid) as p:
                assert f"variant={vid}" in p.describe()
                p.upload(x)
                p.run(steps)
                got = p.download()
            want = oracle.run(L, offs, w, x, steps)
            # 25 steps of at most 13 roundings of 1.1e-16, weights that sum to 1: below 4e-14
            rm, _ = rel_errors(L.interior(got), L.interior(want))
            assert rm <= 1e-12, (ny, nx, halo, steps, rm)
            m = ~L.interior_mask()
            assert np.array_equal(got[m], want[m])


@pytest.mark.parametrize("shape,ny,nx", [("box2d1r", 64, 128), ("box2d1r", 300, 517), ("star2d1r", 31, 300),
                                         ("star2d1r", 700, 127), ("star2d3r", 64, 256), ("star2d3r", 257, 600),
                                         ("box2d1r", 1531, 700)])
def test_default_plans_of_small_grids(gpu, shape, ny, nx):
    # what a plan takes by itself, for step counts that divide evenly or not, against the oracle
    print(f"case {shape} {ny}x{nx}", flush=True)
    r = int(shape[-2])
    offs = shape_offsets(shape)
    L = Layout.with_halo([ny, nx], r)
    w = oracle.fill_weights(len(offs), ny)
    for halo, steps in ((0, 1), (0, 29), (1, 8), (1, 30)):
        x = np.random.default_rng(steps).uniform(-1, 1, L.cells) if halo else oracle.fill_data(L, steps)
        with Plan(L, r, dense_weights(2, r, offs, w), use_graph=bool(steps & 1)) as p:
            p.upload(x)
            p.run(steps)
            p.run(steps)
            got = p.download()
        want = oracle.run(L, offs, w, x, 2 * steps)
        rm, _ = rel_errors(L.interior(got), L.interior(want))
        assert rm <= 1e-12, (halo, steps, rm)
        m = ~L.interior_mask()
        assert np.array_equal(got[m], want[m])
