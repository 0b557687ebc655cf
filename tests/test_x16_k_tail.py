"""The 16x16-block ring kernel's partial last slice: every remainder of k against a 16-byte group, whole k shorter than one group, one
slice and several in front of it, edge tiles, NaN in the padding behind the rows, in every transpose, against the fp64 oracle with the suite's own bounds."""
import numpy as np
import pytest

import util as U

F32, F16 = U.F32, U.F16
NAMES = {F32: "f32", F16: "f16"}
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F32, F16], ids=NAMES.get)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_every_remainder_of_k(dtype, ta, tb):
    import gemm_mmbo_amd as G
    per16, bk = (4, 16) if dtype == F32 else (8, 32)
    info = {c: G.config_info(dtype, c) for c in range(G.num_configs(dtype))}
    ids = [c for c, d in info.items() if "_ACC" in d["name"] and d["split_k"] in (1, 2)]
    assert len(ids) == 16
    for i, cid in enumerate(ids):
        d = info[cid]
        bm, bn = d["macro_tile_m"], d["macro_tile_n"]
        for cut in range(1, per16 + 1):
            slices = (0, 1, 9)[(i + cut) % 3]
            k = slices * bk + ((cut + i) % (bk // per16)) * per16 + cut
            m, n = ((bm, bn), (bm + cut, 2 * bn - 1), (2 * bm - cut, bn + per16))[cut % 3]
            pad, beta = (0, 1, 3)[(i + cut) % 3], (0.0, 0.5)[cut % 2]
            p = U.Problem(dtype, ta, tb, m, n, k, -1.5, beta, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, ldc=m + pad, seed=20 * i + cut,
                          dist="normal" if dtype == F16 else "uniform", c_fill="uniform" if beta else "nan")
            for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
                operand.reshape(-1, ld)[:, rows:] = np.nan
            got, guard = U.run_gpu(p, cid, (cut % 2, i % 2, 0))
            U.check(p, got, f"{d['name']} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{k} pad {pad} beta {beta}")
            assert np.all(guard == 0), "wrote past the end of C"
