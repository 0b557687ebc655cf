"""fp32 products on the bf16 matrix pipes (gemm_planes.hpp): every tile and GlobalSplitU at the edges of tiles and remainders of k, values that
three bf16 planes cannot hold, and the error against 64 bits beside that of the fp32 matrix instructions."""
import numpy as np
import pytest

import util as U

F32 = U.F32
pytestmark = pytest.mark.gpu


TILES = [(256, 128), (128, 128), (128, 64), (64, 64)]       # kPlanesTiles


def _run(p, tile, split, offsets=(0, 0, 0)):
    """The kernel on row `tile` of its tiles, whatever the pick is."""
    import ctypes

    import torch

    import gemm_mmbo_amd as G
    f = G.lib().mmbo_internal_planes_gemm
    sz, ll, vp, ci = ctypes.c_size_t, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int
    f.argtypes = [ci, ci, sz, sz, sz, vp, vp, sz, ll, vp, sz, ll, vp, vp, sz, ll, ci, ci, ci, vp]

    def up(h, off):
        t = torch.zeros(h.size + off + 8, dtype=torch.float32, device="cuda")
        t[off:off + h.size].copy_(torch.from_numpy(h))
        return t
    d = [up(h, off) for h, off in zip((p.A, p.B, p.C), offsets)]
    at = [t.data_ptr() + 4 * off for t, off in zip(d, offsets)]
    al, be = ctypes.c_float(p.alpha), ctypes.c_float(p.beta)
    rc = f(p.ta, p.tb, p.m, p.n, p.k, ctypes.byref(al), at[0], p.lda, p.sa, at[1], p.ldb, p.sb, ctypes.byref(be), at[2], p.ldc, p.sc, p.batch, tile, split, None)
    if rc != 0:
        raise G.MmboError(rc, "planes")
    torch.cuda.synchronize()
    return d[2][offsets[2]:offsets[2] + p.C.size].cpu().numpy(), d[2][offsets[2] + p.C.size:].cpu().numpy()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_edges_of_tiles_and_remainders_of_k(ta, tb):
    """Whole and cut tiles (by one to three rows of a group of four as well), a dimension of four, slices of 32 k whole, cut in and
    between groups of four, one slice to more than the loop's turn holds, columns and padding off 16 bytes, NaN in the padding."""
    for i in range(20):
        tile, split = i % 4, (1, 2, 4, 8, 16)[i // 4]
        bm, bn = TILES[tile]
        for j, (m, n) in enumerate(((bm, bn), (bm + 1, 2 * bn - 1), (2 * bm - 2, bn + 3), (4, bn + 2), (bm + 3, 4))):
            k = (32, 37, 64, 95, 4, 129, 318, 96, 33, 226, 61, 160)[(i + 5 * j) % 12] * (1, split)[j % 2]
            pad, beta = (0, 1, 4)[(i + j) % 3], (0.0, 0.5)[(i // 4 + j) % 2]
            p = U.Problem(F32, ta, tb, m, n, k, -1.5, beta, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, ldc=m + pad, seed=20 * i + j,
                          c_fill="uniform" if beta else "nan")
            for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
                operand.reshape(-1, ld)[:, rows:] = np.nan
            got, guard = _run(p, tile, split, (j % 2, i % 2, j % 3))
            U.check(p, got, f"{bm}x{bn} split {split} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{k} pad {pad} beta {beta}")
            assert np.all(guard == 0), "wrote past the end of C"


def test_a_contiguous_dimension_shorter_than_a_load_is_refused():
    import gemm_mmbo_amd as G
    for ta, tb, m, n, k in ((0, 0, 3, 64, 64), (1, 1, 64, 3, 64), (0, 0, 64, 64, 3), (0, 0, 64, 64, 0)):
        p = U.Problem(F32, ta, tb, m, n, k, seed=1)
        for tile in range(4):
            with pytest.raises(G.MmboError) as e:
                _run(p, tile, 1)
            assert e.value.status == 5
        for cid in range(G.num_configs(F32)):
            if "_BF16X3" in G.config_info(F32, cid)["name"]:
                with pytest.raises(G.MmboError) as e:
                    U.run_gpu(p, cid)
                assert e.value.status == 5


def test_batches_and_the_config_ids():
    """Strided batches (a problem to an XCD, and not), every GlobalSplitU, and the ids of the tiles that have some."""
    import gemm_mmbo_amd as G
    for tile, (bm, bn) in enumerate(TILES):
        for batch, split in ((8, 1), (3, 1), (3, 4)):
            p = U.Problem(F32, tile % 2, split % 2, bm + 5, bn + 9, 200, 1.0, 1.0, batch=batch, ldc=bm + 7, seed=tile + batch + split)
            got, guard = _run(p, tile, split)
            U.check(p, got, f"{bm}x{bn} batch {batch} split {split}")
            assert np.all(guard == 0)
    ids = {c: d for c in range(G.num_configs(F32)) if "_BF16X3" in (d := G.config_info(F32, c))["name"]}
    assert len(ids) == 10
    for cid, d in ids.items():
        p = U.Problem(F32, 0, 1, 300, 200, 700, 1.0, 0.5, seed=cid)
        named, direct = U.run_gpu(p, cid)[0], _run(p, TILES.index((d["macro_tile_m"], d["macro_tile_n"])), d["split_k"])[0]
        U.check(p, named, d["name"])
        assert np.array_equal(named, direct), d["name"]


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_values_that_three_planes_cannot_hold(ta, tb):
    """Infinities, NaN, elements that round up to a bf16 infinity, sums that overflow, elements whose lower planes fall below bf16's
    smallest number (beside small and large ones) or that vanish: what the fp32 matrix instructions give, to an fp32 sum's error."""
    m, n, k = 150, 140, 70
    f = np.float32
    cases = {
        "inf": lambda a, b: (a.__setitem__((3, 5), np.inf), a.__setitem__((149, 69), -np.inf), b.__setitem__((7, 139), np.inf)),
        "inf times zero": lambda a, b: (a.__setitem__((3, 5), np.inf), b.__setitem__((5, slice(0, 70)), 0)),
        "nan": lambda a, b: a.__setitem__((0, 0), np.nan),
        "largest": lambda a, b: (a.__setitem__((10, 20), np.finfo(f).max), b.__setitem__((20, slice(None)), f(2.0) ** -100)),
        "overflow": lambda a, b: (a.__setitem__((10, slice(None)), f(3e38)), b.__imul__(np.sign(b))),      # (of one sign: else it is a matter of order)
        "small": lambda a, b: a.__imul__(f(2.0) ** -118),
        "small times large": lambda a, b: (a.__imul__(f(2.0) ** -120), b.__imul__(f(2.0) ** 90)),
        "subnormal": lambda a, b: a.__imul__(f(1e-41)),
        "zeros": lambda a, b: a.__imul__(f(0)),
        "one small row": lambda a, b: a.__setitem__(100, a[100] * f(2.0) ** -115),
    }
    for name, spoil in cases.items():
        p = U.Problem(F32, ta, tb, m, n, k, seed=len(name))
        a = p.A.reshape((k, m) if ta else (m, k), order="F").T.copy() if ta else p.A.reshape((m, k), order="F").copy()
        b = p.B.reshape((n, k), order="F").T.copy() if tb else p.B.reshape((k, n), order="F").copy()
        spoil(a, b)
        p.A = np.asfortranarray(a.T if ta else a).reshape(-1, order="F").copy()
        p.B = np.asfortranarray(b.T if tb else b).reshape(-1, order="F").copy()
        with np.errstate(all="ignore"):
            want = a.astype(np.float64) @ b.astype(np.float64)
            terms = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
        for tile, split in [(t, s) for t in range(4) for s in (1, 2)]:
            got = _run(p, tile, split)[0].reshape((m, n), order="F").astype(np.float64)
            label = f"{name}: {TILES[tile]} split {split}"
            over = np.abs(want) > np.finfo(f).max                   # (and infinities of the fp64 sum)
            assert np.array_equal(np.isnan(got), np.isnan(want)), label
            assert np.array_equal(got[over], np.sign(want[over]) * np.inf), label
            ok = np.isfinite(want) & ~over
            # k roundings, each of at most half an ulp: 2^-24 of the terms' sum, or 2^-150 where the sum is below the smallest normal number
            assert np.all(np.abs(got[ok] - want[ok]) <= k * (2.0 ** -24 * terms[ok] + 2.0 ** -150)), label


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_one_small_column(ta, tb):
    """A column of B whose lower planes fall below bf16's smallest number, beside ordinary ones: each place that a column can have among the four that a
    lane holds."""
    m, n, k = 150, 140, 70
    for col in (0, 1, 2, 3, 77, 138):
        p = U.Problem(F32, ta, tb, m, n, k, seed=col)
        a = p.A.reshape((k, m) if ta else (m, k), order="F").T if ta else p.A.reshape((m, k), order="F")
        b = p.B.reshape((n, k), order="F").T.copy() if tb else p.B.reshape((k, n), order="F").copy()
        b[:, col] *= np.float32(2.0) ** -122
        p.B = np.asfortranarray(b.T if tb else b).reshape(-1, order="F").copy()
        want = a.astype(np.float64) @ b.astype(np.float64)
        # k roundings, each of at most half an ulp: 2^-24 of the terms' sum, or 2^-150 where the sum is below the smallest normal number
        bound = k * (2.0 ** -24 * (np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))) + 2.0 ** -150)
        for tile, split in [(t, s) for t in range(4) for s in (1, 2)]:
            got = _run(p, tile, split)[0].reshape((m, n), order="F").astype(np.float64)
            off = np.abs(got - want) > bound
            assert not off.any(), f"column {col}: {TILES[tile]} split {split}: {np.argwhere(off)[:3].tolist()}, {got[off][:3]} not {want[off][:3]}"


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_elements_that_planes_lose_beside_ordinary_ones(ta, tb):
    """Elements that vanish in three planes, or leave nothing of a sum, in some rows or columns of tiles whose other sums are ordinary: such a sum
    is an exact zero.  (Below 2^-134 an element vanishes, below 2^-109 it loses bits.)"""
    m, n, k = 150, 140, 70
    two = np.float32(2.0)

    def pair(a, b):                       # 2^-120 (1 + 2^-20) - 2^-120, the first one's tail below the planes
        a[33] = 0
        a[33, 1], a[33, 40] = two ** -120 * (1 + two ** -20), -(two ** -120)
        b[1], b[40] = two ** 100, two ** 100
    cases = {                             # what is done to op(A) and op(B)
        "vanishing row": lambda a, b: (a.__setitem__(7, np.sign(a[7]) * two ** -136), b.__imul__(two ** 100)),
        "vanishing column": lambda a, b: (b.__setitem__((slice(None), 77), np.sign(b[:, 77]) * two ** -138), a.__imul__(two ** 100)),
        "vanishing row beside an ordinary operand": lambda a, b: a.__setitem__(149, np.float32(1e-41)),
        "last column of a cut tile": lambda a, b: (b.__setitem__((slice(None), 139), np.float32(1e-42)), a.__imul__(two ** 90)),
        "one element beside zeros": lambda a, b: (a.__setitem__(64, 0), a.__setitem__((64, 69), np.float32(1e-41)), b.__imul__(np.float32(1e30))),
        "subnormal row": lambda a, b: (a.__setitem__(130, a[130] * two ** -127), b.__imul__(two ** 60)),
        "zero rows and columns": lambda a, b: (a.__setitem__(slice(20, 90), 0), b.__setitem__((slice(None), slice(60, 140)), 0)),
        "cancelling pair": pair,
    }
    for name, spoil in cases.items():
        p = U.Problem(F32, ta, tb, m, n, k, seed=len(name))
        a = p.A.reshape((k, m) if ta else (m, k), order="F").T.copy() if ta else p.A.reshape((m, k), order="F").copy()
        b = p.B.reshape((n, k), order="F").T.copy() if tb else p.B.reshape((k, n), order="F").copy()
        spoil(a, b)
        p.A = np.asfortranarray(a.T if ta else a).reshape(-1, order="F").copy()
        p.B = np.asfortranarray(b.T if tb else b).reshape(-1, order="F").copy()
        want = a.astype(np.float64) @ b.astype(np.float64)
        # k roundings, each of at most half an ulp: 2^-24 of the terms' sum, or 2^-150 where the sum is below the smallest normal number
        bound = k * (2.0 ** -24 * (np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))) + 2.0 ** -150)
        if name == "cancelling pair":
            bound[33] = 0                 # (two products and their sum, all of them fp32 numbers)
        for tile, split in [(t, s) for t in range(4) for s in (1, 2)]:
            got = _run(p, tile, split)[0].reshape((m, n), order="F").astype(np.float64)
            off = np.abs(got - want) > bound
            assert not off.any(), f"{name}: {TILES[tile]} split {split}: {np.argwhere(off)[:3].tolist()}, {got[off][:3]} not {want[off][:3]}"


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_tiles_that_are_computed_again(ta, tb):
    """A NaN in every tile: the other rows come from the fp32 MFMAs, in steps of 16 k whole and cut, tiles cut by the edge, NaN in the padding."""
    for tile, (bm, bn) in enumerate(TILES):
        for i, k in enumerate((4, 15, 16, 17, 31, 33, 64, 79, 130, 208)):
            m, n, split, pad = bm + (5, 3, 62)[i % 3], (bn + 3, bn - 1)[i % 2], (1, 2)[i // 5 % 2], (0, 1, 4)[i % 3]
            p = U.Problem(F32, ta, tb, m, n, k, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, seed=10 * tile + i)
            for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
                operand.reshape(-1, ld)[:, rows:] = np.nan
            stored_a, stored_b = p.A.reshape(-1, p.lda)[:, :k if ta else m], p.B.reshape(-1, p.ldb)[:, :n if tb else k]     # (column by column)
            a, b = stored_a if ta else stored_a.T, stored_b.T if not tb else stored_b
            spoiled = (3, bm + 1)
            for row in spoiled:
                for q in range(0, k, 32 * ((k + 63) // 64)):          # (in every split)
                    a[row, q] = np.nan
            others = [r for r in range(m) if r not in spoiled]
            got, guard = _run(p, tile, split, (i % 2, i // 2 % 2, i % 3))
            got = got.reshape((m, n), order="F").astype(np.float64)
            label = f"{bm}x{bn} split {split} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{k} pad {pad}"
            assert np.isnan(got[list(spoiled)]).all() and np.all(guard == 0), label
            x, y = a[others].astype(np.float64), b.astype(np.float64)
            # k roundings, each of at most half an ulp of the terms' sum
            assert np.all(np.abs(got[others] - x @ y) <= k * 2.0 ** -24 * (np.abs(x) @ np.abs(y))), label


def test_what_a_tile_that_is_computed_again_costs():
    """NN 1024^3 with a NaN in every tile, beside the same call without: 2.4 times the time, 8.5 where elements are fetched one by one."""
    import torch

    import gemm_mmbo_amd as G
    n = 1024
    assert "_BF16X3" in G.auto_info(F32, 0, 0, n, n, n)["name"]
    A = [torch.rand(n * n, device="cuda") * 2 - 1 for _ in range(2)]
    A[1].view(n, n)[0, ::64] = float("nan")
    B, C = torch.rand(n * n, device="cuda") * 2 - 1, torch.empty(n * n, device="cuda")
    best = [float("inf")] * 2
    for _ in range(8):
        for q in range(2):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            G.gemm(F32, 0, 0, n, n, n, 1.0, A[q], n, B, n, 0.0, C, n)
            start.record()
            for _ in range(20):
                G.gemm(F32, 0, 0, n, n, n, 1.0, A[q], n, B, n, 0.0, C, n)
            end.record()
            end.synchronize()
            best[q] = min(best[q], start.elapsed_time(end))
    assert best[1] < 4 * best[0], best


def test_not_less_exact_than_the_fp32_matrix_instructions():
    """2-norm of the error against 64 bits, on the same operands: one run of k in planes beside one run of fp32 matrix instructions.  Uniform,
    positive and widely spread operands."""
    import gemm_mmbo_amd as G
    native = next(c for c in range(G.num_configs(F32)) if "_ACC" in (d := G.config_info(F32, c))["name"] and d["macro_tile_m"] == d["macro_tile_n"] == 128)
    m = n = 192
    for dist in ("uniform", "positive", "spread"):
        for k in (64, 100, 600, 3000):
            p = U.Problem(F32, 1, 0, m, n, k, seed=k)
            if dist == "positive":
                p.A, p.B = np.abs(p.A), np.abs(p.B)
            if dist == "spread":
                rng = np.random.default_rng(k)
                p.A = (p.A * 2.0 ** rng.uniform(-20, 20, p.A.shape)).astype(np.float32)
                p.B = (p.B * 2.0 ** rng.uniform(-20, 20, p.B.shape)).astype(np.float32)
            want = p.exact().reshape(-1, order="F")

            def error(got):
                return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))
            limit = error(U.run_gpu(p, native)[0])
            for tile in range(4):
                here = error(_run(p, tile, 1)[0])
                assert here <= limit, (dist, k, TILES[tile], here, limit)


def test_sums_of_few_terms():
    """A weighted gather and its like: op(A) with one, two or sixteen elements that are not zero in a row.  From two terms on not less exact than the fp32 matrix
    instructions; a single product lacks x2*y3 + x3*y2 + x3*y3, at most (2 * 2^-8 * 2^-16 + 2^-32) of it, beside one rounding of half a unit, 2^-24 of it."""
    import gemm_mmbo_amd as G
    native = next(c for c in range(G.num_configs(F32)) if "_ACC" in (d := G.config_info(F32, c))["name"] and d["macro_tile_m"] == d["macro_tile_n"] == 128)
    m, n, k = 512, 384, 256
    for terms in (1, 2, 16):
        p = U.Problem(F32, 1, 0, m, n, k, seed=terms)
        a = p.A.reshape(m, k)
        np.put_along_axis(a, np.argsort(np.random.default_rng(terms).random((m, k)), axis=1)[:, terms:], 0, axis=1)
        want = p.exact().reshape(-1, order="F")
        native_off, off = (x[0].astype(np.float64) - want for x in (U.run_gpu(p, native), _run(p, 1, 1)))
        if terms > 1:
            assert np.linalg.norm(off) <= np.linalg.norm(native_off), terms
        else:
            assert np.all(np.abs(off) <= (2.0 ** -23 + 2.0 ** -32 + 2.0 ** -24) * np.abs(want))
            # (1.017 is measured on a million products; these are 200,000)
            assert np.linalg.norm(off) <= 1.03 * np.linalg.norm(native_off)


def test_a_cut_group_of_rows_costs_no_round_trips_of_its_own():
    """NT 1639 x 1845 x 256 with beta, whose last group of four rows has three, beside 1640 rows in the same operands: 1.0 times the time; 1.3 where the old C of
    such a group is requested element by element as it is used."""
    import torch

    import gemm_mmbo_amd as G
    ld, n, k = 1640, 1845, 256
    A, B, C = (torch.rand(x, device="cuda") for x in (ld * k, n * k, ld * n))
    best = {1639: float("inf"), 1640: float("inf")}
    assert all("_BF16X3" in G.auto_info(F32, 0, 1, m, n, k, lda=ld, ldc=ld, reads_c=True)["name"] for m in best)
    for _ in range(10):
        for m in best:
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            G.gemm(F32, 0, 1, m, n, k, -1.0, A, ld, B, n, 0.5, C, ld)
            start.record()
            for _ in range(50):
                G.gemm(F32, 0, 1, m, n, k, -1.0, A, ld, B, n, 0.5, C, ld)
            end.record()
            end.synchronize()
            best[m] = min(best[m], start.elapsed_time(end))
    assert best[1639] < 1.15 * best[1640], best


def test_tiles_that_are_computed_again_are_as_exact():
    """A NaN in every tile, the error of the other rows against 64 bits beside that of eight runs of fp32 matrix instructions (1,024 k each), on operands of one
    sign, where it grows with a run's length."""
    import gemm_mmbo_amd as G
    native = next(c for c in range(G.num_configs(F32)) if "_ACC" in (d := G.config_info(F32, c))["name"] and d["macro_tile_m"] == d["macro_tile_n"] == 128 and d["split_k"] == 8)
    m, n, k = 256, 128, 8192
    p = U.Problem(F32, 1, 0, m, n, k, seed=5)
    p.A, p.B = np.abs(p.A), np.abs(p.B)
    p.A.reshape(m, k)[::64, 0] = np.nan
    rows = np.arange(m) % 64 != 0
    want = (p.B.reshape(n, k).astype(np.float64) @ p.A.reshape(m, k)[rows].astype(np.float64).T)

    def error(got):
        return float(np.linalg.norm(got.reshape(n, m)[:, rows] - want) / np.linalg.norm(want))
    limit = error(U.run_gpu(p, native)[0])
    for tile in range(4):
        here = error(_run(p, tile, 1)[0])
        assert here <= limit, (TILES[tile], here, limit)
