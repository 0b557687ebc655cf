"""fp64 problems whose last 64 x 64 tiles go out as quarters (tests/util.py holds the tolerance): grids just past a whole round
of 256 tiles, at the rule's edges, with edge tiles that fill one, two or all four quarters."""
import numpy as np
import pytest

import util as U

pytestmark = pytest.mark.gpu

TILE_64, TILE_128x64 = 2, 5          # rows of the fp64 config table


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,beta,ldc", [
    (1024, 1024, 48, 1.0, 0),          # 256 tiles: none quartered
    (257 * 64, 64, 32, 0.0, 0),        # 257: one tile, all four quarters whole
    (16385, 33, 33, 1.0, 16390),       # 257: one row and 33 columns in the last tile, odd k
    (1087, 1000, 20, 0.5, 0),          # 272: edge tiles of 63 rows and 40 columns among the quartered ones
    (448 * 64, 40, 17, 1.0, 0),        # 448 = 256 + 192: the most
    (449 * 64, 40, 17, 0.0, 0),        # 449: none
    (1152, 2048, 7, -1.0, 1160),       # 576, less than a stage of k
])
def test_quartered_tiles(ta, tb, m, n, k, beta, ldc):
    p = U.Problem(U.F64, ta, tb, m, n, k, -1.0, beta, ldc=ldc or None, seed=m + n + k, c_fill="nan" if beta == 0.0 else "uniform")
    got, guard = U.run_gpu(p, TILE_64, (0, 0, 0))
    U.check(p, got, f"{m}x{n}x{k}")
    assert np.all(guard == 0), "wrote past the end of C"
    # every element's sum runs over k in the same order whatever the tile
    whole, _ = U.run_gpu(p, TILE_128x64, (0, 0, 0))
    assert got.tobytes() == whole.tobytes()
