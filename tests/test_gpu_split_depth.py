"""Split precision, 49-point box: the default plans' depth-6 launches give the bits of depth 2."""
import numpy as np
import pytest

from convstencil_amd import Plan, Layout, shape_offsets, dense_weights
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp16w3", "bf16x3"])
# partial and single tiles, and one grid of the size that takes the larger tile
@pytest.mark.parametrize("ny,nx,steps", [(1, 1, 7), (64, 64, 6), (77, 131, 11), (300, 517, 10), (65, 200, 15),
                                         (3001, 4003, 17)])
def test_depth_gives_the_same_bits(gpu, prec, ny, nx, steps):
    print(f"case {prec} {ny}x{nx} T={steps}", flush=True)
    offs = shape_offsets("box2d3r")
    w = dense_weights(2, 3, offs, oracle.fill_weights(len(offs), ny))
    L = Layout.with_halo([ny, nx], 3)
    got = []
    for depth in (0, 2):
        with Plan(L, 3, w, precision=prec, fusion_depth=depth) as p:
            p.fill_random(nx)
            assert p.run(steps).fusion_depth == (6 if depth == 0 else 2)
            got.append(p.download())
    # the two round alike except where the FP64 sum of a depth-2 launch's last step is itself a tie
    # between two FP32 numbers: fewer than one cell in a million
    assert np.count_nonzero(got[0] != got[1]) <= 1e-6 * L.cells
    assert np.max(np.abs(got[0] - got[1])) <= 1e-7
