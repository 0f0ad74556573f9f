"""The split 2-D kernels' column offset CS: the narrowest tile that keeps every block's reads inside, except
for the kernels whose anchors lie where depth 2 has them (staging 3), which only default plans take."""
import ctypes

import pytest

from convstencil_amd import _lib
from test_kernel_emulation import ctable


def _variants():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    lib.cs_debug_variant_info.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                                          ctypes.c_char_p, ctypes.c_int32]
    out = []
    for i in range(lib.cs_debug_variant_count(4)):
        info = (ctypes.c_int64 * 12)()
        lib.cs_debug_variant_info(4, i, info, None, 0)
        v = dict(zip(("id", "prec", "R", "shape", "kf", "by", "bx", "nw", "lds", "px", "st", "cs"), map(int, info)))
        if v["st"] >= 2:
            out.append(v)
    return out


VARIANTS = _variants()


def _least(v):
    c0, _, tx, _ = ctable(v["R"], v["shape"])
    for cs in range(64):
        lo = [v["R"] * (s + 1) for s in range(v["kf"])]
        if min(x - (x + cs + c0) % 8 + min(tx) for x in lo) + cs >= 0:
            return cs


@pytest.mark.parametrize("v", VARIANTS, ids=[str(v["id"]) for v in VARIANTS])
def test_column_offset(v):
    if v["st"] == 2:
        assert v["cs"] == _least(v)
        return
    two = next(u for u in VARIANTS if u["st"] == 2 and (u["prec"], u["R"], u["shape"], u["kf"]) == (v["prec"], 3, 0, 2))
    assert (v["R"], v["shape"], v["kf"] % 2) == (3, 0, 0) and v["kf"] > 2
    assert (3 * v["kf"] + v["cs"]) % 8 == (6 + two["cs"]) % 8 and v["cs"] >= _least(v)


def test_no_kernel_with_depth_2_anchors_in_fp16x2():
    # its plans take depth 2, so no depth of it has to agree with that one
    assert {v["prec"] for v in VARIANTS if v["st"] == 3} == {1, 4}
