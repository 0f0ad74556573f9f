"""The stacked-wave 3-D FP64 kernels (k3d_tile.hip) against the CPU oracle: every variant at the tile's
own size, one cell more, several tiles and z chunks; and what plans take by themselves."""
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
    for i in range(lib.cs_debug_variant_count(13)):
        info = (ctypes.c_int64 * 12)()
        name = ctypes.create_string_buffer(128)
        lib.cs_debug_variant_info(13, i, info, name, 128)
        out.append((int(info[0]), "star" if info[3] else "box", int(info[4]), int(info[5]), name.value.decode()))
    return out


VARIANTS = _variants()


@pytest.mark.parametrize("vid,kind,kf,by,name", VARIANTS, ids=[v[4] for v in VARIANTS])
def test_every_tile_variant(gpu, vid, kind, kf, by, name):
    print(f"case {name}", flush=True)
    offs = shape_offsets(f"{kind}3d1r")
    w = oracle.fill_weights(len(offs), vid)
    for k, n in enumerate([[1, by, 64], [2, by + 1, 65], [7, 2 * by - 2 * kf, 128 - 2 * kf],
                           [45, 2 * by - 2 * kf + 1, 131]]):
        L = Layout.with_halo(n, 1 + (k & 1), k)
        x = oracle.fill_data(L, vid + k)
        for steps in (kf, 2 * kf + 1):
            with Plan(L, 1, dense_weights(3, 1, offs, w), variant=vid) as p:
                assert f"variant={vid}" in p.describe()
                p.upload(x)
                p.run(steps)
                got = p.download()
            want = oracle.run(L, offs, w, x, steps)
            # 9 steps of at most 27 roundings of 1.1e-16, weights that sum to 1: below 3e-14
            rm, _ = rel_errors(L.interior(got), L.interior(want))
            assert rm <= 1e-12, (n, steps, rm)
            m = ~L.interior_mask()
            assert np.array_equal(got[m], want[m])


@pytest.mark.parametrize("shape", ["box3d1r", "star3d1r"])
@pytest.mark.parametrize("n", [[5, 24, 64], [70, 23, 64], [70, 24, 63], [9, 200, 150], [130, 67, 90]])
def test_default_plans(gpu, shape, n):
    # at and just below the smallest tile, with zero and with alternating halos
    print(f"case {shape} {n}", flush=True)
    offs = shape_offsets(shape)
    L = Layout.with_halo(n, 1)
    w = oracle.fill_weights(len(offs), sum(n))
    for halo, steps in ((0, 1), (0, 2), (0, 11), (1, 5)):
        x = np.random.default_rng(steps).uniform(-1, 1, L.cells) if halo else oracle.fill_data(L, steps)
        with Plan(L, 1, dense_weights(3, 1, offs, w), use_graph=bool(steps & 1)) as p:
            assert ("mf=12" in p.describe()) == (n[1] >= 24 and n[2] >= 64)
            p.upload(x)
            p.run(steps)
            p.run(steps)
            got = p.download()
        want = oracle.run(L, offs, w, x, 2 * steps)
        rm, _ = rel_errors(L.interior(got), L.interior(want))
        assert rm <= 1e-12, (halo, steps, rm)
        m = ~L.interior_mask()
        assert np.array_equal(got[m], want[m])
