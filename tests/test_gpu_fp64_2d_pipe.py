"""The level-pipelined 2-D FP64 kernels (k2d_pipe_body.h) against the CPU oracle, at the sizes where
their strips, chunks and pipelines can go wrong, with zero and non-zero halos."""
import ctypes

import numpy as np
import pytest

from convstencil_amd import Plan, Layout, shape_offsets, dense_weights, _lib
from oracle import oracle
from refimpl import rel_errors
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


def _variants():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    lib.cs_debug_variant_count.restype = ctypes.c_int32
    lib.cs_debug_variant_info.restype = ctypes.c_int32
    lib.cs_debug_variant_info.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                                          ctypes.c_char_p, ctypes.c_int32]
    out = []
    for fam in (10, 11):
        for i in range(lib.cs_debug_variant_count(fam)):
            info = (ctypes.c_int64 * 12)()
            name = ctypes.create_string_buffer(128)
            lib.cs_debug_variant_info(fam, i, info, name, 128)
            out.append((int(info[0]), int(info[2]), "star" if info[3] else "box", int(info[4]), int(info[6]),
                        name.value.decode()))
    return out


VARIANTS = _variants()


def _check(L, got, want):
    # 1e-12 relative max: at most 2 * 7 * 7 roundings of 1.1e-16 per step and 2 kf + 3 <= 35 steps
    # of weights that sum to 1 give 3.8e-13
    rm, _ = rel_errors(L.interior(got), L.interior(want))
    assert rm <= 1e-12, rm


# one strip of exactly 512 columns; two strips that overlap almost wholly; a strip boundary (512
# + ox columns: two strips without slack, one more: three); one row; fewer rows than the depth
SIZES = [(1, 512, 0), (5, 513, 1), (40, "b", 0), (37, "b+1", 3), (300, 1100, 0)]


@pytest.mark.parametrize("vid,r,kind,kf,ox,name", VARIANTS, ids=[v[5] for v in VARIANTS])
def test_every_pipe_variant(gpu, vid, r, kind, kf, ox, name):
    shape = f"{kind}2d{r}r"
    offs = shape_offsets(shape)
    for k, (ny, nx, pad) in enumerate(SIZES):
        nx = 512 + ox + (nx != "b") if isinstance(nx, str) else nx
        print(f"case {name} {ny}x{nx} pad {pad}", flush=True)
        L = Layout.with_halo([ny, nx], r + (k & 1), pad)
        w = oracle.fill_weights(len(offs), vid + k)
        x = oracle.fill_data(L, vid + k)
        steps = 2 * kf + 3  # fused launches and a remainder
        with Plan(L, r, dense_weights(2, r, offs, w), variant=vid) as p:
            assert f"variant={vid}" in p.describe()
            p.upload(x)
            p.run(steps)
            got = p.download()
        want = oracle.run(L, offs, w, x, steps)
        _check(L, got, want)
        m = ~L.interior_mask()
        assert not got[m].any()  # the halo is never written


@pytest.mark.parametrize("vid,r,kind,kf,ox,name", VARIANTS, ids=[v[5] for v in VARIANTS])
def test_pipe_variant_uniform_halo(gpu, vid, r, kind, kf, ox, name):
    # the same non-zero halo in both buffers, in caller-owned buffers: the general halo form, on
    # outer and on inner strips' edge chunks, against the oracle's fixed halo
    print(f"case {name} uniform halo", flush=True)
    shape = f"{kind}2d{r}r"
    offs = shape_offsets(shape)
    ny, nx = 70, 512 + 2 * ox
    L = Layout.with_halo([ny, nx], r)
    w = oracle.fill_weights(len(offs), vid)
    x = np.random.default_rng(vid).uniform(-1, 1, L.cells)
    steps = kf
    hip = _Hip()
    a, b = hip.alloc(x.nbytes), hip.alloc(x.nbytes)
    try:
        hip.h2d(a, x)
        hip.h2d(b, x)
        d = np.ascontiguousarray(dense_weights(2, r, offs, w))
        st = _lib.cs_stencil(2, r, d.ctypes.data_as(_lib.c_double_p))
        opt = _lib.cs_options()
        opt.tile_variant = vid
        fin = ctypes.c_int32(-1)
        Lc = L.to_c()
        assert _lib.load().cs_run_2d_noalloc(ctypes.byref(Lc), ctypes.byref(st), a, b, steps, ctypes.byref(opt), None,
                                             ctypes.byref(fin)) == _lib.CS_OK
        assert hip.lib.hipDeviceSynchronize() == 0
        got = np.empty_like(x)
        hip.d2h(got, b if fin.value else a)
    finally:
        hip.lib.hipFree(a)
        hip.lib.hipFree(b)
    # fixed halo: step the oracle one step at a time, putting the halo back
    want = x.copy()
    m = L.interior_mask()
    for _ in range(steps):
        nxt = oracle.run(L, offs, w, want, 1)
        want[m] = nxt[m]
    _check(L, got, want)
    assert np.array_equal(got[~m], x[~m])


def test_narrow_grids_refuse_a_pipe_variant(gpu):
    # 511 columns: no strip fits; a forced variant is refused, the default plan runs
    offs = shape_offsets("box2d1r")
    L = Layout.with_halo([40, 511], 1)
    d = dense_weights(2, 1, offs, oracle.fill_weights(len(offs), 3))
    with pytest.raises(_lib.ConvStencilError):
        Plan(L, 1, d, variant=901012)
    with Plan(L, 1, d) as p:
        assert "k2d_pipe" not in p.describe()


@pytest.mark.parametrize("vid,r,kind,kf,ox,name", VARIANTS, ids=[v[5] for v in VARIANTS])
def test_pipe_variant_alternating_halo(gpu, vid, r, kind, kf, ox, name):
    # an uploaded non-zero halo and a zeroed second buffer: every level reads the halo of the
    # buffer that its step of the ping-pong reads, for odd and even counts of launches, split
    # launches, single-step ends and runs that continue one another
    print(f"case {name} alternating halo", flush=True)
    offs = shape_offsets(f"{kind}2d{r}r")
    L = Layout.with_halo([70, 512 + ox + 9], r, 2)
    w = oracle.fill_weights(len(offs), vid)
    x = np.random.default_rng(vid).uniform(-1, 1, L.cells)
    for runs in ((kf,), (2 * kf,), (kf + 3,), (2 * kf + 1, 3 * kf), (3,)):
        with Plan(L, r, dense_weights(2, r, offs, w), variant=vid, use_graph=len(runs) > 1) as p:
            p.upload(x)
            for s in runs:
                p.run(s)
            got = p.download()
        want = oracle.run(L, offs, w, x, sum(runs))
        _check(L, got, want)
        m = ~L.interior_mask()
        assert np.array_equal(got[m], want[m]), runs


PIPES = [v for v in VARIANTS if v[5].startswith("k2d_pipe")]


@pytest.mark.parametrize("vid,r,kind,kf,ox,name", PIPES, ids=[v[5] for v in PIPES])
def test_pipe_variant_long_chunks_halo(gpu, vid, r, kind, kf, ox, name):
    # 40000 rows on two strips: chunks of 150 rows and more, so that the ring of the side halos (64 rows)
    # wraps and the loop without row checks runs long in the general halo form.  Windows of 1000 rows far from
    # the first and last row against the oracle on their rows and those that they depend on
    print(f"case {name} long chunks", flush=True)
    offs = shape_offsets(f"{kind}2d{r}r")
    ny, nx, steps = 40000, 512 + ox, 2 * kf
    L = Layout.with_halo([ny, nx], r)
    w = oracle.fill_weights(len(offs), vid)
    x = np.random.default_rng(vid).uniform(-1, 1, L.cells)
    with Plan(L, r, dense_weights(2, r, offs, w), variant=vid) as p:
        assert f"variant={vid}" in p.describe()
        p.upload(x)
        p.run(steps)
        got = p.download()
    n, reach = 1000, r * steps
    sub = Layout.with_halo([n + 2 * reach, nx], r)
    pitch = sub.cells // (n + 2 * reach + 2 * r)
    assert L.cells == (ny + 2 * r) * pitch
    X, G = x.reshape(-1, pitch), got.reshape(-1, pitch)
    for row in (700, 20011, ny - 1900):
        part = X[row - reach : row + n + reach + 2 * r]
        want = oracle.run(sub, offs, w, np.ascontiguousarray(part).ravel(), steps).reshape(-1, pitch)
        want = want[r + reach : r + reach + n]
        have = G[r + row : r + row + n]
        assert np.abs(have[:, r : r + nx] - want[:, r : r + nx]).max() <= 1e-12 * np.abs(want).max(), row
        assert np.array_equal(have[:, :r], want[:, :r]) and np.array_equal(have[:, r + nx :], want[:, r + nx :])


@pytest.mark.parametrize("ny,nx,strips", [(9700, 520, True), (2600, 2500, True), (2000, 7600, False)])
def test_depth_12_box_by_halo(gpu, ny, nx, strips):
    # depth 12 asked for, the radius-1 box: strips of that depth with a zero halo where they are faster (10000 x 520,
    # 48 steps, 281 us against the pipeline's 348), the pipeline with an uploaded halo
    print(f"case depth 12 {ny}x{nx}", flush=True)
    offs = shape_offsets("box2d1r")
    L = Layout.with_halo([ny, nx], 1)
    w = oracle.fill_weights(len(offs), ny)
    zero = oracle.fill_data(L, ny)
    halo = np.random.default_rng(ny).uniform(-1, 1, L.cells)
    with Plan(L, 1, dense_weights(2, 1, offs, w), fusion_depth=12) as p:
        for x in (zero, halo, zero):
            p.upload(x)
            family = "k2d_reg" if strips and x is zero else "k2d_pipe"
            assert f"name={family}" in p.describe()
            for s in (12, 20, 11):
                p.run(s)
            got = p.download()
            _check(L, got, oracle.run(L, offs, w, x, 43))
