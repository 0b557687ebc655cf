"""fp64 operands at every alignment on the loader that tests no chunk: even and odd row counts past the last whole tile, odd leading
dimensions and pointers, whole and partial stages of k.  NaN in the rows between the matrix and its leading dimension: what
a repeated row brings in, or the second half of a pair that an odd count of rows ends in, may not reach a stored element."""
import numpy as np
import pytest

import util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,pad,offsets,beta", [
    (130, 66, 48, 0, (0, 0, 0), 1.0),          # even edges, whole stages
    (131, 67, 53, 0, (0, 0, 0), 0.0),          # odd edges, odd leading dimensions, a partial stage
    (256, 128, 32, 1, (0, 0, 0), 1.0),         # whole tiles of odd leading dimensions
    (258, 129, 17, 3, (1, 1, 1), 0.5),         # off 16 bytes everywhere
    (2, 1, 64, 5, (1, 0, 1), 1.0),             # one pair of rows, one column
    (131, 67, 48, 0, (0, 0, 0), 1.0),          # odd edges, whole stages only: the last one holds the column with nothing behind it
    (129, 33, 32, 2, (0, 1, 0), 0.5),          # ... with a padding row behind each column but the last
    (1, 1, 49, 0, (0, 0, 0), 1.0),             # one row: every pair takes in the next column
    (1, 3, 16, 0, (1, 1, 1), 0.0),             # ... one stage, whose last column goes element by element
])
def test_every_config_unaligned(ta, tb, m, n, k, pad, offsets, beta):
    import gemm_mmbo_amd as G
    p = U.Problem(U.F64, ta, tb, m, n, k, 1.5, beta, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, ldc=m + pad,
                  seed=m + n + k + pad, c_fill="nan" if beta == 0.0 else "uniform")
    for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
        operand.reshape(-1, ld)[:, rows:] = np.nan
    for cid in range(G.num_configs(U.F64)):
        got, guard = U.run_gpu(p, cid, offsets)
        U.check(p, got, f"cfg {cid}")
        assert np.all(guard == 0), "wrote past the end of C"
