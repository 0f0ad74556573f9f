"""FP64 batches on the register-tile kernels: several grids' tiles in one launch, mixed with grids too
small for a tile, against the CPU oracle."""
import numpy as np
import pytest

from convstencil_amd import Batch, Layout, shape_offsets, dense_weights
from oracle import oracle
from refimpl import rel_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
# the tiles' own sizes, one cell less and more, several tiles; one and more launches
@pytest.mark.parametrize("steps", [1, 2, 13, 40])
def test_batch_of_tiles(gpu, graph, steps):
    print(f"case T={steps} graph={graph}", flush=True)
    grids = [("box2d1r", 32, 128), ("box2d1r", 31, 128), ("box2d1r", 32, 127), ("box2d1r", 33, 129),
             ("box2d1r", 150, 301), ("box2d1r", 64, 128), ("star2d3r", 64, 256),
             ("star2d3r", 63, 256), ("star2d3r", 65, 257), ("star2d3r", 200, 531), ("star2d3r", 5, 7)]
    Ls, ws, ds, xs = [], [], [], []
    for i, (s, ny, nx) in enumerate(grids):
        offs = shape_offsets(s)
        Ls.append(Layout.with_halo([ny, nx], int(s[-2])))
        ws.append(oracle.fill_weights(len(offs), i))
        ds.append(dense_weights(2, int(s[-2]), offs, ws[-1]))
        xs.append(oracle.fill_data(Ls[-1], i))
    with Batch(Ls, [int(s[-2]) for s, _, _ in grids], ds, use_graph=graph) as b:
        for i, x in enumerate(xs):
            b.upload(i, x)
        b.run(steps)
        b.run(steps)
        got = [b.download(i) for i in range(len(grids))]
    for i, (s, ny, nx) in enumerate(grids):
        want = oracle.run(Ls[i], shape_offsets(s), ws[i], xs[i], 2 * steps)
        # 80 steps of at most 13 roundings of 1.1e-16, weights that sum to 1: below 2e-13
        rm, _ = rel_errors(Ls[i].interior(got[i]), Ls[i].interior(want))
        assert rm <= 1e-12, (s, ny, nx, rm)
        m = ~Ls[i].interior_mask()
        assert np.array_equal(got[i][m], want[m])
