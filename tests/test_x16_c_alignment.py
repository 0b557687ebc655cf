"""The 16x16-block ring kernel's epilogue where the columns of C start at any element: whole tiles and edge tiles, with the old C fetched
under the last slices (fp16), requested ahead, or not read, columns on odd elements, in every transpose, against the fp64 oracle with the suite's own bounds."""
import numpy as np
import pytest

import util as U

F32, F16 = U.F32, U.F16
NAMES = {F32: "f32", F16: "f16"}
pytestmark = pytest.mark.gpu


def _ids(dtype):
    """One id per tile, without a split of k."""
    import gemm_mmbo_amd as G
    info = {c: G.config_info(dtype, c) for c in range(G.num_configs(dtype))}
    return [c for c, d in info.items() if "_ACC" in d["name"] and d["split_k"] == 1]


@pytest.mark.parametrize("dtype", [F32, F16], ids=NAMES.get)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_columns_of_c_at_any_element(dtype, ta, tb):
    import gemm_mmbo_amd as G
    g, bk = (4, 16) if dtype == F32 else (8, 32)
    ids = _ids(dtype)
    assert len(ids) == 8
    for i, cid in enumerate(ids):
        d = G.config_info(dtype, cid)
        bm, bn = d["macro_tile_m"], d["macro_tile_n"]
        #        m          n       slices  ldc - m  offset of C
        cases = [(bm, bn, 8, 1, 1), (2 * bm, bn, 3, g // 2, 0), (bm, 2 * bn, 9, 0, g - 1),             # whole tiles
                 (bm + g, bn + 1, 8, 3, 1), (bm + g - 1, bn + g, 3, 0, 0),                            # the cut group one row long, all but one
                 (2 * bm - 1, bn + 3, 2, 1, 0), (g, bn - 1, 8, 1, 3),
                 # columns on odd elements of a C that starts on a dword: every length of the cut group, whole tiles, over a batch
                 (2 * bm, bn + 1, 3, 1, 0)] + [(bm // 2 + 2 * g + r, bn - 2, 2, 1 - (g + r) % 2, 0) for r in range(g)] + [(g + 1, g + 2, 2, 0, 0)]
        for q, (m, n, slices, more, offset) in enumerate(cases):
            alpha, beta, batch = (1.0, -1.5)[(i + q) % 2], (0.0, 0.5, 1.0)[(i + q) % 3], 1 + (q in (3, 7))
            p = U.Problem(dtype, ta, tb, m, n, bk * slices, alpha, beta, ldc=m + more, batch=batch, seed=60 * i + q,
                          dist="normal" if dtype == F16 else "uniform", c_fill="uniform" if beta else "nan")
            got, guard = U.run_gpu(p, cid, (0, 0, offset))
            U.check(p, got, f"{d['name']} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{bk * slices} beta {beta} ldc {m + more} offset {offset}")
            assert np.all(guard == 0), "wrote past the end of C"


def test_every_column_of_c_on_an_odd_element():
    """fp16, C on an odd element and an even leading dimension: every length of the group that an edge cuts, whole tiles, a batch, beta on and
    off; the element in front of C, whose dword the first column shares, stays as it is."""
    import torch

    import gemm_mmbo_amd as G
    for i, cid in enumerate(_ids(F16)):
        d = G.config_info(F16, cid)
        bm, bn = d["macro_tile_m"], d["macro_tile_n"]
        shapes = [(bm // 2 + 16 + r, bn - 2 + r % 3, 1) for r in range(8)] + [(2 * bm, bn, 1), (9, 10, 1), (5, bn, 1), (bm + 3, bn + 1, 3)]
        for q, (m, n, batch) in enumerate(shapes):
            ta, tb, beta = 1 if m < 8 else (i + q) % 2, (q // 2) % 2, (0.5, 0.0, 1.0)[(i + q) % 3]     # (no row-contiguous A of fewer than 8 rows)
            p = U.Problem(F16, ta, tb, m, n, 64 + 8 * (q % 2), 1.0, beta, ldc=m + m % 2, batch=batch, seed=30 * i + q, dist="normal",
                          c_fill="uniform" if beta else "nan")
            got, guard = U.run_gpu(p, cid, (0, 0, 1))
            U.check(p, got, f"{d['name']} {'NT'[ta]}{'NT'[tb]} {m}x{n} batch {batch} beta {beta}")
            assert np.all(guard == 0), "wrote past the end of C"
        m, n, k = bm + 5, bn, 64
        A, B = (torch.ones(count, device="cuda", dtype=torch.float16) for count in (m * k, k * n))
        C = torch.full(((m + m % 2) * n + 2,), -7.0, device="cuda", dtype=torch.float16)
        G.gemm(F16, 0, 0, m, n, k, 1.0, A, m, B, k, 0.5, C.data_ptr() + 2, m + m % 2, cid)
        torch.cuda.synchronize()
        assert float(C[0]) == -7.0 and float(C[-1]) == -7.0
        want = torch.full((n, m + m % 2), k - 3.5, device="cuda", dtype=torch.float16)
        want[:, m:] = -7.0
        assert torch.equal(C[1:-1].view(n, m + m % 2), want)
