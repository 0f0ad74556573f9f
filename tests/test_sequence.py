"""The launch sequences of default 2-D FP64 plans (cs_sequence.cpp), on the host: they make the steps, end in
the buffer that single steps would end in, and take the family that measured faster where lines by
the grid's size alone had taken another."""
import ctypes

import pytest

from convstencil_amd import _lib

BOX, STAR = 0, 1
MFMA, STRIP, PIPE, TILE = 4, 7, 10, 11


def _lib_():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    lib.cs_debug_sequence_2d.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.c_int64, ctypes.c_int64, ctypes.c_int32,
                                         ctypes.c_int64, ctypes.POINTER(ctypes.c_int32),
                                         ctypes.POINTER(ctypes.c_int64), ctypes.c_int32]
    lib.cs_debug_variant_info.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                                          ctypes.c_char_p, ctypes.c_int32]
    return lib


LIB = _lib_()


def _variants():
    out = {}
    for family in (2, 8, 10, 11, 12):
        for i in range(LIB.cs_debug_variant_count(family)):
            info = (ctypes.c_int64 * 12)()
            LIB.cs_debug_variant_info(family, i, info, None, 0)
            out[int(info[0])] = dict(zip(("mf", "R", "shape", "kf", "by", "bx", "nw", "lds", "px"), map(int, info[1:10])))
    return out


VARIANTS = _variants()


def _sequence(R, shape, ny, nx, zero, steps):
    ids, counts = (ctypes.c_int32 * 80)(), (ctypes.c_int64 * 80)()
    n = LIB.cs_debug_sequence_2d(R, shape, ny, nx, zero, steps, ids, counts, 80)
    assert n >= 0
    return [(VARIANTS[ids[i]], counts[i]) for i in range(n)]


GRIDS = [(1, 512), (32, 128), (33, 129), (64, 256), (63, 600), (97, 4001), (300, 517), (1531, 2749), (2048, 2048),
         (20000, 520), (520, 20000), (4096, 4096), (10240, 10240), (3, 100000)]


@pytest.mark.parametrize("R,shape", [(1, BOX), (1, STAR), (3, STAR), (3, BOX)])
@pytest.mark.parametrize("zero", [1, 0])
def test_steps_and_buffers(R, shape, zero):
    covered = 0
    for ny, nx in GRIDS:
        for steps in list(range(1, 70)) + [127, 128, 129, 1000, 100001]:
            seq = _sequence(R, shape, ny, nx, zero, steps)
            if not seq:
                continue
            covered += 1
            assert sum(v["kf"] * n for v, n in seq) == steps
            ended = False  # single-step kernels read their input buffer's halo: they come last
            for v, n in seq:
                assert (v["R"], v["shape"]) == (R, shape) and n > 0
                assert v["mf"] != PIPE or nx >= 64 * v["px"]
                assert v["mf"] != TILE or (ny >= v["by"] and nx >= v["bx"])
                if not zero:
                    assert v["mf"] in (PIPE, TILE) or (v["mf"], v["kf"]) == (MFMA, 1)
                    assert not ended or v["mf"] == MFMA
                    ended = v["mf"] == MFMA
            if not zero:
                assert sum(n for _, n in seq) % 2 == steps % 2
    assert covered > 200


def test_other_stencils_and_empty_grids_keep_their_rule():
    assert not _sequence(2, BOX, 1000, 1000, 1, 10)
    assert not _sequence(3, BOX, 1000, 511, 1, 10)
    assert not _sequence(1, BOX, 0, 1000, 1, 10)
    assert not _sequence(1, STAR, 31, 127, 1, 10)


# us of the whole run: what a line by the number of cells took, and the family that was faster
@pytest.mark.parametrize("R,shape,ny,nx,zero,steps,family", [
    (3, STAR, 27884, 520, 1, 48, STRIP),   # pipelines 1204, strips 966
    (3, STAR, 40000, 1000, 1, 48, STRIP),  # pipelines 2331, strips 2191
    (3, BOX, 27884, 520, 1, 48, MFMA),     # pipelines 3189, tables 2703
    (3, STAR, 300, 517, 1, 1, MFMA),       # tiles 13.0, tables 6.4
    (3, BOX, 4096, 4096, 1, 1, MFMA),      # strips 131, tables 74
    (3, BOX, 4096, 4096, 1, 3, MFMA),      # strips and pipelines 245, tables 172
    (3, STAR, 4096, 4096, 1, 4, STRIP),    # pipelines 88.5, strips 76.5
    (3, STAR, 700, 700, 0, 1, MFMA),       # tiles 23.7, tables 6.8
    (1, BOX, 700, 700, 0, 1, MFMA),        # tiles 7.1, tables 6.1
    (3, BOX, 20000, 700, 0, 1, MFMA),      # strips 194, tables 61
])
def test_the_faster_family(R, shape, ny, nx, zero, steps, family):
    assert {v["mf"] for v, _ in _sequence(R, shape, ny, nx, zero, steps)} == {family}


@pytest.mark.parametrize("ny,nx", [(3500, 1000), (2333, 1500), (1590, 2200), (875, 4000)])
def test_no_shallow_tiles(ny, nx):
    # radius-3 star, 48 steps: tiles so shallow that each CU has one, 948-1017 us; strips 459-473
    assert all(v["kf"] >= 4 for v, _ in _sequence(3, STAR, ny, nx, 1, 48))


@pytest.mark.parametrize("shape", [BOX, STAR])
def test_3d_steps(shape):
    # every number of steps from 2 up is made of launches of 2 to 4: none is left for the single-step
    # kernel (star 30 x 24 x 1000, 3 steps: 2 + 1 72 us, the strips before them 32)
    LIB.cs_debug_sequence_3d.argtypes = [ctypes.c_int32, ctypes.c_int32] + [ctypes.c_int64] * 4 + [
        ctypes.POINTER(ctypes.c_int32), ctypes.POINTER(ctypes.c_int64), ctypes.c_int32]
    depth = {}
    for i in range(LIB.cs_debug_variant_count(13)):
        info = (ctypes.c_int64 * 12)()
        LIB.cs_debug_variant_info(13, i, info, None, 0)
        depth[int(info[0])] = (int(info[3]), int(info[4]), int(info[5]), int(info[6]))
    ids, counts = (ctypes.c_int32 * 8)(), (ctypes.c_int64 * 8)()
    for n in ([1, 24, 64], [30, 24, 1000], [17, 90, 130], [100, 100, 100], [512, 512, 512], [3, 3000, 3000]):
        for steps in list(range(2, 40)) + [1000, 100001]:
            k = LIB.cs_debug_sequence_3d(1, shape, *n, steps, ids, counts, 8)
            assert k > 0
            got = [(depth[ids[i]], counts[i]) for i in range(k)]
            assert sum(v[1] * c for v, c in got) == steps
            assert all(v[0] == shape and v[2] <= n[1] and v[3] <= n[2] and c > 0 for v, c in got)
    assert LIB.cs_debug_sequence_3d(1, shape, 10, 23, 64, 4, ids, counts, 8) == 0
    assert LIB.cs_debug_sequence_3d(2, shape, 100, 100, 100, 4, ids, counts, 8) == 0


def _batch_tiles(R, shape, sizes, steps):
    fn = LIB.cs_debug_batch_tiles
    fn.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                   ctypes.POINTER(ctypes.c_int64), ctypes.c_int64]
    col = (ctypes.c_int64 * len(sizes))
    return fn(R, shape, len(sizes), col(*[s[0] for s in sizes]), col(*[s[1] for s in sizes]), steps)


@pytest.mark.parametrize("R,shape,sizes,steps,tiles", [
    (3, STAR, [(2500, 2500)], 60, False),  # 1029 us on tiles, 864 in strips
    (3, STAR, [(1200, 1100), (900, 1000), (700, 1400), (1500, 1100)], 60, False),  # 4.7 M cells: 881 / 715
    (3, STAR, [(900, 1000), (700, 1000), (1000, 1000)], 1, False),  # 94 / 51
    (3, STAR, [(600, 500)] * 3, 60, True),  # 0.9 M cells: 305 / 620
    (1, BOX, [(2500, 2500)], 60, True),  # 360 / 526
    (1, BOX, [(1000, 1000)] * 10, 60, True),  # 10 M cells: 601 / 850
    (3, STAR, [(63, 300)], 60, False),  # smaller than a tile
])
def test_batch_tiles(R, shape, sizes, steps, tiles):
    assert (_batch_tiles(R, shape, sizes, steps) > 0) == tiles
