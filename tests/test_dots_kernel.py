"""The fp64 kernel for small results of long sums (gemm_dots.hpp): every tile at its edges, steps of 32 k whole and cut, runs of a wavefront
shorter and longer than its ring, and where the automatic pick takes it."""
import ctypes

import numpy as np
import pytest

import util as U

F64 = U.F64
INVALID_SIZE, INVALID_CONFIG = 3, 5                           # mmbo_status
TILES = [(4, 4), (4, 8), (8, 4), (8, 8), (8, 16), (16, 8)]      # kDotsTiles


def _call(ta, tb, m, n, k, alpha, A, lda, sa, B, ldb, sb, beta, C, ldc, sc, batch, tile):
    import gemm_mmbo_amd as G
    f = G.lib().mmbo_internal_dots_gemm
    sz, ll, vp, ci = ctypes.c_size_t, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int
    f.argtypes = [ci, ci, sz, sz, sz, vp, vp, sz, ll, vp, sz, ll, vp, vp, sz, ll, ci, ci, vp]
    al, be = ctypes.c_double(alpha), ctypes.c_double(beta)
    return f(ta, tb, m, n, k, ctypes.byref(al), A, lda, sa, B, ldb, sb, ctypes.byref(be), C, ldc, sc, batch, tile, None)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_edges_of_tiles_steps_and_rings(ta, tb):
    """Whole tiles, tiles cut to every count of rows and of columns, problems of fewer rows than a tile; operands and C from odd
    elements, NaN in the padding and right behind it; batches."""
    import torch
    for tile, (bm, bn) in enumerate(TILES):
        for j, k in enumerate((1, 31, 32, 33, 63, 255, 256, 257, 511, 2047, 2304, 2305, 2623, 4129)):
            m = (2 * bm, bm + 1 + j % (bm - 1), 2 + j % bm, bm)[j % 4]
            n = (bn, 2 + j % bn, 2 * bn, 9 * bn + 1 + j % (bn - 1))[(j + j // 4) % 4]
            pad, beta, batch = (0, 1, 3)[j % 3], (0.0, 0.5)[j % 2], (1, 1, 1, 3)[j % 4]
            p = U.Problem(F64, ta, tb, m, n, k, -1.5, beta, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, ldc=m + pad, batch=batch,
                          seed=20 * tile + j, c_fill="uniform" if beta else "nan")
            for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
                operand.reshape(-1, ld)[:, rows:] = np.nan
            d = []
            for h, off in ((p.A, j % 2), (p.B, tile % 2), (p.C, 1)):
                t = torch.full((h.size + off + 8,), float("nan"), dtype=torch.float64, device="cuda")
                t[off:off + h.size].copy_(torch.from_numpy(h))
                d.append((t, off))
            at = [t.data_ptr() + 8 * off for t, off in d]
            assert _call(ta, tb, m, n, k, p.alpha, at[0], p.lda, p.sa, at[1], p.ldb, p.sb, p.beta, at[2], p.ldc, p.sc, batch, tile) == 0
            torch.cuda.synchronize()
            got = d[2][0][1:1 + p.C.size].cpu().numpy()
            U.check(p, got, f"{bm}x{bn} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{k} pad {pad} beta {beta} batch {batch}")
            assert bool(d[2][0][1 + p.C.size:].isnan().all()) and bool(d[2][0][:1].isnan().all()), "wrote outside C"


def test_a_row_contiguous_operand_of_one_row_is_refused():
    """Its loads take two rows; the automatic pick leaves such calls to the kernels that take any."""
    one = 16                                                    # (never dereferenced: refused before anything is launched)
    for tile in range(len(TILES)):
        assert _call(0, 0, 1, 64, 4096, 1.0, one, 1, 0, one, 4096, 0, 0.0, one, 1, 0, 1, tile) == INVALID_SIZE
        assert _call(1, 1, 64, 1, 4096, 1.0, one, 4096, 0, one, 1, 0, 0.0, one, 64, 0, 1, tile) == INVALID_SIZE
    assert _call(1, 0, 64, 64, 4096, 1.0, one, 4096, 0, one, 4096, 0, 0.0, one, 64, 0, 1, len(TILES)) == INVALID_CONFIG


@pytest.mark.parametrize("ta,tb,m,n,k,lda,taken", [
    (1, 0, 49, 45, 57216, 57216, True), (0, 1, 49, 45, 57216, 49, True), (0, 0, 34, 48, 20000, 64, True),
    (0, 0, 1, 4096, 4096, 1, False),                            # one row, row-contiguous
    (1, 0, 2048, 2048, 2048, 2048, False), (0, 1, 44160, 2048, 384, 44160, False), (0, 0, 512, 512, 512, 512, False),
    (1, 0, 49, 45, 57216, 1 << 24, None),                       # 16 columns of A span 2 GiB: no kernel takes it
])
def test_where_the_automatic_pick_takes_it(ta, tb, m, n, k, lda, taken):
    import gemm_mmbo_amd as G
    if taken is None:
        with pytest.raises(G.MmboError):
            G.auto_info(F64, ta, tb, m, n, k, lda=lda)
        return
    info = G.auto_info(F64, ta, tb, m, n, k, lda=lda)
    assert ("DOTS" in info["name"]) == taken, info["name"]
    if taken:
        assert info["split_k"] == 1 and info["threads"] == 512 and info["lds_bytes"] <= 160 * 1024


def test_nothing_else_reads_the_direct_loads_register(tmp_path):
    """The direct loads are asm statements that change M0 without saying so: only they, and the s_mov in front of each, may name it; and
    scratch memory would put loads of the compiler's own between them."""
    import os

    import test_kernel_asm as K
    if not os.path.exists(K.HIPCC):
        pytest.skip("hipcc not installed")
    path = K._compile(("inst_dots.hip", ["-DMMBO_TILE=3"]), str(tmp_path))
    kernels = {name: body for name, body in K._kernels(path).items() if any(t.startswith("v_mfma") for t in body)}
    assert len(kernels) == 4
    for name, body in kernels.items():
        loads = [t for t in body if t.startswith("buffer_load_dwordx4") and "lds" in t]
        assert loads and len([t for t in body if t.startswith("s_mov_b32 m0")]) == len(loads), name
        assert not [t for t in body if " m0" in t and not t.startswith("s_mov_b32 m0")], name
        assert not [t for t in body if t.startswith("scratch_")], name
