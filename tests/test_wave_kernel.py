"""The split-by-wavefront kernel (csrc/gemm_wave.hpp), which the automatic pick takes for small, thin and long-k problems.

GPU: every (element type, tile, transposes) the library ships, named through an entry point of the tests' own, with one, four and
eight wavefronts, with and without GlobalSplitU, at sizes around the tile, around the ring's depth of slices (odd and even runs, a
partial slice), at every alignment, with NaN in the padding rows; the walks of the grid that only whole memory lines
take; and small, thin and long-k shapes through the automatic pick (rows shorter than a 16-byte group, fewer slices than wavefronts,
GlobalSplitU beyond 16, where several threads share the splits of one sum).  All against the fp64 oracle with the suite's own
bounds.  CPU: facts about the generated code that the kernel's asm statements rely on.
"""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

import util as U

F32, F16, F64 = U.F32, U.F16, U.F64
NAMES = {F32: "f32", F16: "f16", F64: "f64"}
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gemm_mmbo_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

#         m    n     k    batch  what it is there for
SHAPES = [(1, 1, 64, 1), (1, 130, 33, 1), (7, 3, 515, 1), (3, 257, 96, 1),           # rows shorter than a 16-byte group
          (15, 17, 31, 1), (16, 16, 32, 1), (17, 15, 64, 1), (31, 33, 128, 3), (33, 31, 129, 8),
          (63, 65, 160, 1), (65, 63, 255, 5), (128, 96, 1, 2), (40, 56, 9, 1),
          (20, 12, 8192, 1), (12, 700, 3001, 1), (700, 12, 3001, 1), (64, 48, 40000, 1), (5, 9, 65537, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, F16, F64], ids=NAMES.get)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_small_thin_and_long_k_shapes(dtype, ta, tb):
    import torch

    import gemm_mmbo_amd as G
    taken = 0
    for i, (m, n, k, batch) in enumerate(SHAPES):
        pad = (0, 1, 8)[i % 3]
        ar, br = U.stored_shape(ta, m, k)[0], U.stored_shape(tb, k, n)[0]
        p = U.Problem(dtype, ta, tb, m, n, k, -1.5, (0.0, 0.5)[i % 2], lda=ar + pad, ldb=br + pad, ldc=m + pad, batch=batch,
                      seed=300 + i, dist="normal" if dtype == F16 else "uniform", c_fill=("nan", "uniform")[i % 2])
        got, guard = U.run_gpu(p)
        taken += G.auto_info(dtype, ta, tb, m, n, k, batch, p.lda, p.ldb, p.ldc, p.beta != 0)["config_id"] == -1
        U.check(p, got, f"{NAMES[dtype]} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{k} b{batch}")
        assert np.all(guard == 0)
        # the entry point that allocates nothing: the same bits
        dA, dB, dC = (torch.from_numpy(x).cuda() for x in (p.A, p.B, p.C))
        G.gemm_strided_batched_static_workspace(dtype, ta, tb, m, n, k, -1.5, dA, p.lda, p.sa, dB, p.ldb, p.sb, p.beta, dC, p.ldc,
                                                p.sc, batch)
        torch.cuda.synchronize()
        assert np.array_equal(dC.cpu().numpy().view(U.BITS[dtype]), got.view(U.BITS[dtype]))
    assert 2 * taken >= len(SHAPES)               # (the others run a config: the shapes are the same for every type)


#        rows, columns, slices in the ring
TILES = [(16, 16, 8), (16, 32, 6), (32, 16, 6), (16, 64, 4), (64, 16, 4), (32, 32, 4), (32, 64, 4), (64, 32, 4)]
BK = {F32: 16, F16: 32, F64: 8}
SHIPPED = [(dtype, tile) for dtype in (F32, F16, F64) for tile in range(6 if dtype == F64 else len(TILES))]


def _wave_gemm(p, tile, waves, split, offset_elems=(0, 0, 0)):
    """The problem on one instantiation of the kernel; returns C and the words behind it, or None where there is none."""
    import torch

    import gemm_mmbo_amd as G
    L = G.lib()
    f = L.mmbo_internal_wave_gemm
    f.restype = ctypes.c_int
    f.argtypes = L.mmbo_gemm_strided_batched.argtypes[:-2] + [ctypes.c_int] * 3 + [ctypes.c_void_p]
    dev = []
    for h, off in zip((p.A, p.B, p.C), offset_elems):
        t = torch.zeros(h.size + off + 8, dtype={F32: torch.float32, F16: torch.float16, F64: torch.float64}[p.dtype], device="cuda")
        t[off:off + h.size].copy_(torch.from_numpy(h))
        dev.append((t, t.data_ptr() + off * U.ESZ[p.dtype]))
    scalar = ctypes.c_double if p.dtype == F64 else ctypes.c_float
    alpha, beta = scalar(p.alpha), scalar(p.beta)
    rc = f(p.dtype, p.ta, p.tb, p.m, p.n, p.k, ctypes.byref(alpha), dev[0][1], p.lda, p.sa, dev[1][1], p.ldb, p.sb, ctypes.byref(beta),
           dev[2][1], p.ldc, p.sc, p.batch, tile, waves, split, None)
    if rc == 5:                                  # no such instantiation
        return None
    assert rc == 0, rc
    torch.cuda.synchronize()
    out = dev[2][0].cpu().numpy()
    return out[offset_elems[2]:offset_elems[2] + p.C.size], out[offset_elems[2] + p.C.size:]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, F16, F64], ids=NAMES.get)
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_every_instantiation(dtype, tile):
    bm, bn, depth = TILES[tile]
    bk, ran = BK[dtype], 0
    for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
        for waves in (1, 4, 8):
            for split in (1, 5):
                if split > 1 and dtype == F64:
                    continue
                # (m, n, k, padding rows, offsets, batch): edges, an odd run of slices and a partial one; whole tiles, a full ring
                # and one pair more; edges packed tightly, where the last columns have nothing behind them, over a batch
                cases = [(bm - 1, bn + 1, (depth + 1) * bk * waves * split + 3, 1 + tile % 3, (1, 1, 1), 1),
                         (2 * bm, bn, (depth + 2) * bk * waves * split, 0, (0, 0, 0), 1),
                         (bm + 1, 2 * bn - 1, bk * waves * split + bk, 0, (0, 1, 0), 3)]
                for i, (m, n, k, pad, offsets, batch) in enumerate(cases):
                    beta = (0.5, 0.0, 1.0)[i]
                    p = U.Problem(dtype, ta, tb, m, n, k, -1.5, beta, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, ldc=m + pad,
                                  batch=batch, seed=40 * tile + i, dist="normal" if dtype == F16 else "uniform",
                                  c_fill="uniform" if beta else "nan")
                    for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
                        operand.reshape(-1, ld)[:, rows:] = np.nan
                    got = _wave_gemm(p, tile, waves, split, offsets)
                    if got is None:
                        continue
                    ran += 1
                    U.check(p, got[0], f"{NAMES[dtype]} tile {tile} {'NT'[ta]}{'NT'[tb]} w{waves} s{split} {m}x{n}x{k}")
                    assert np.all(got[1] == 0), "wrote past the end of C"
    waves = 3 if 8 * depth * (bm + bn) * 64 <= 160 * 1024 else 2
    assert ran == (4 * 3 * waves * (1 if dtype == F64 else 2) if (dtype, tile) in SHIPPED else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tile", SHIPPED, ids=lambda v: str(v))
def test_groups_that_an_edge_cuts(dtype, tile):
    """16-byte groups cut by the end of k, of a row-contiguous operand, or of a column of C that is read come as the 16 bytes that end there:
    every length of the cut group, operands shorter than one group, NaN in the padding behind."""
    bm, bn, _ = TILES[tile]
    bk, per16 = BK[dtype], 16 // U.ESZ[dtype]
    q = 0
    for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
        for cut in range(1, per16 + 1):
            waves, pad = (1, 4, 8)[q % 3], (0, 1, 3)[q % 3]
            if waves > 1 and 8 * TILES[tile][2] * (bm + bn) * 64 > 160 * 1024:
                waves = 4
            cases = [(bm + cut, bn + 1, 2 * bk * waves + cut, 1), (cut, 2 * bn - 1, bk + per16 + cut, 2), (bm - cut, cut, cut, 3),
                     (bm + 1, bn + cut, 4 * bk * waves + 2 * bk - cut, 1)]
            for i, (m, n, k, batch) in enumerate(cases):
                beta = (0.5, 1.0, -1.0, 0.0)[i]
                p = U.Problem(dtype, ta, tb, m, n, k, (1.0, -1.5)[i % 2], beta, lda=(k if ta else m) + pad, ldb=(n if tb else k) + pad, ldc=m + pad,
                              batch=batch, seed=10 * q + i, dist="normal" if dtype == F16 else "uniform", c_fill="uniform" if beta else "nan")
                for operand, ld, rows in ((p.A, p.lda, k if ta else m), (p.B, p.ldb, n if tb else k)):
                    operand.reshape(-1, ld)[:, rows:] = np.nan
                got = _wave_gemm(p, tile, waves, 1, (q % 2, i % 2, (q + i) % 2))
                assert got is not None
                U.check(p, got[0], f"{NAMES[dtype]} tile {tile} {'NT'[ta]}{'NT'[tb]} w{waves} {m}x{n}x{k} pad {pad}")
                assert np.all(got[1] == 0), "wrote past the end of C"
            q += 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tile,ta,tb,m,n,k,lda,ldb", [
    (F32, 5, 0, 1, 576, 1792, 105, 640, 1856),       # longer side of whole lines across: tile rows first
    (F16, 6, 0, 1, 65, 1024, 96, 128, 1024),         # ... two tile rows, the second nearly empty
    (F32, 7, 0, 0, 2048, 70, 80, 2048, 81),          # longer side down: the dispatcher's order
    (F64, 0, 0, 0, 256, 16, 40, 256, 40),            # ... one tile column
    (F32, 5, 1, 1, 100, 70, 64, 64, 71),             # regrouped by XCD
])
def test_walks_of_the_grid(dtype, tile, ta, tb, m, n, k, lda, ldb):
    p = U.Problem(dtype, ta, tb, m, n, k, 1.0, 0.5, lda=lda, ldb=ldb, ldc=m + 3, seed=tile + m, dist="normal" if dtype == F16 else "uniform")
    got, guard = _wave_gemm(p, tile, 4, 1)
    U.check(p, got, f"{NAMES[dtype]} tile {tile}")
    assert np.all(guard == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_operands_whose_slices_span_two_gigabytes_take_a_config(ta, tb):
    """A pair of slices must fit a buffer descriptor: the automatic pick leaves the kernel where the leading dimension is too large."""
    import torch

    import gemm_mmbo_amd as G
    m, n, k, ld = 64, 64, 20, 2 ** 31 // (32 * 4) + 64
    lda, ldb = (k if ta else ld), (ld if tb else k)
    assert G.auto_info(F32, ta, tb, m, n, k)["config_id"] == -1
    huge = (lda == ld) or (ldb == ld)
    assert (G.auto_info(F32, ta, tb, m, n, k, lda=lda, ldb=ldb)["config_id"] >= 0) == huge
    rng = np.random.default_rng(5)
    hA, hB = rng.uniform(-1, 1, (k, m)).astype(np.float32), rng.uniform(-1, 1, (k, n)).astype(np.float32)

    def stored(h, rows_contiguous, ld):                       # h: k x rows
        h = h if rows_contiguous else h.T.copy()
        t = torch.zeros((h.shape[0] - 1) * ld + h.shape[1], dtype=torch.float32, device="cuda")
        for i in range(h.shape[0]):
            t[i * ld:i * ld + h.shape[1]] = torch.from_numpy(h[i])
        return t
    dA, dB = stored(hA, not ta, lda), stored(hB, bool(tb), ldb)
    dC = torch.full((m * n,), float("nan"), dtype=torch.float32, device="cuda")
    G.gemm(F32, ta, tb, m, n, k, 1.0, dA, lda, dB, ldb, 0.0, dC, m)
    torch.cuda.synchronize()
    want = hA.T.astype(np.float64) @ hB.astype(np.float64)
    assert np.max(np.abs(dC.cpu().numpy().reshape((m, n), order="F") - want)) <= U.tol(F32, k) * max(np.max(np.abs(want)), 1.0)


@pytest.mark.gpu
def test_only_calls_whose_pick_splits_k_take_a_workspace():
    """mmbo_select_config tells a caller whether a call uses a workspace (before a capture, or beside another call of the entry
    point that allocates nothing): with GlobalSplitU 1, and so for every fp64 call, none may be taken."""
    import torch

    import gemm_mmbo_amd as G
    split = 0
    for dtype in (F32, F16, F64):
        t = {F32: torch.float32, F16: torch.float16, F64: torch.float64}[dtype]
        for (ta, tb, m, n, k) in ((0, 0, 64, 489, 4640), (1, 0, 336, 448, 11520), (0, 1, 32, 48, 30000), (0, 0, 700, 12, 3001),
                                  (0, 0, 40, 9000, 700), (1, 1, 100, 300, 2100), (0, 0, 500, 400, 600)):
            dA, dB, dC = (torch.zeros(c, device="cuda", dtype=t) for c in (m * k, k * n, m * n))
            torch.cuda.synchronize()
            G.release_workspace()
            G.gemm(dtype, ta, tb, m, n, k, 1.0, dA, k if ta else m, dB, n if tb else k, 0.0, dC, m)
            torch.cuda.synchronize()
            splits = G.config_info(dtype, G.select_config(dtype, ta, tb, m, n, k, 1))["split_k"] > 1
            split += splits
            assert splits or G.workspace_info()[0] == 0, (NAMES[dtype], ta, tb, m, n, k)
    assert split > 0
    G.release_workspace()


#            dtype ta tb  m    n      k       whose plans differ with beta or with padded leading dimensions
REPLANNED = [(F16, 0, 0, 520, 608, 3968), (F32, 0, 1, 128, 10200, 2176), (F32, 0, 0, 32, 4863, 10379), (F16, 0, 0, 192, 2298, 8384),
             (F32, 0, 1, 1856, 32, 10384), (F32, 1, 0, 32, 5454, 9120), (F16, 0, 1, 64, 48, 40000)]


def _variants(ta, tb, m, n, k):
    """(lda, ldb, beta) of calls of one shape: packed without C first."""
    a, b = (k if ta else m), (n if tb else k)
    return [(a, b, 0.0), (a, b, 1.0), (a + 1, b + 1, 0.0), (a + 8, b + 8, 1.0), (-(-a // 64) * 64, -(-b // 64) * 64, 1.0)]


def test_whether_k_is_split_over_work_groups_follows_from_the_shape():
    """No call of a shape whose packed call without C needs no workspace needs one, and none needs more than that call leaves behind (at
    least 8 MiB where it needs one)."""
    import random

    import gemm_mmbo_amd as G

    def need(dtype, ta, tb, m, n, k, lda, ldb, beta):
        info = G.auto_info(dtype, ta, tb, m, n, k, 1, lda, ldb, None, beta != 0.0)
        return (info["split_k"] * m * n * 4 if info["split_k"] > 1 else 0), info["config_id"]
    rng, seen = random.Random(4), 0
    shapes = list(REPLANNED)
    while len(shapes) < 1500:
        thin, wide, k = int(2 ** rng.uniform(3, 9)), int(2 ** rng.uniform(3, 13)), int(2 ** rng.uniform(9, 16))
        shapes.append((rng.choice((F32, F16)), rng.randint(0, 1), rng.randint(0, 1)) + rng.choice(((thin, wide, k), (wide, thin, k))))
    for shape in shapes:
        ta, tb, m, n, k = shape[1:]
        packed, *others = [need(*shape, *v) for v in _variants(ta, tb, m, n, k)]
        for bytes_needed, _ in others:
            assert bytes_needed <= (max(packed[0], 8 << 20) if packed[0] else 0), shape
        # a call that names the pick of mmbo_select_config leaves enough behind as well
        split = G.config_info(shape[0], G.select_config(*shape))["split_k"]
        assert packed[0] <= (max(split * m * n * 4, 8 << 20) if split > 1 else 0), shape
        seen += len({o[0] for o in [packed] + others}) > 1
    assert seen > 0                                   # (plans do differ between the calls of a shape)


@pytest.mark.gpu
def test_one_call_of_a_shape_leaves_the_workspace_of_all():
    """Run once, then captured with another beta or other leading dimensions: nothing is allocated, and each replay of the graph gives
    the bits of the eager call."""
    import torch

    import gemm_mmbo_amd as G
    stream = torch.cuda.Stream()
    for shape in REPLANNED:
        dtype, ta, tb, m, n, k = shape
        t = {F32: torch.float32, F16: torch.float16}[dtype]
        variants = _variants(ta, tb, m, n, k)
        with torch.cuda.stream(stream):
            gen = torch.Generator(device="cuda")
            gen.manual_seed(7)
            dA = torch.rand(max(v[0] for v in variants) * (m if ta else k), device="cuda", generator=gen).mul_(0.1).to(t)
            dB = torch.rand(max(v[1] for v in variants) * (k if tb else n), device="cuda", generator=gen).mul_(0.1).to(t)
            C0 = torch.rand(m * n, device="cuda", generator=gen).to(t)
            dC = C0.clone()

            def call(lda, ldb, beta):
                G.gemm(dtype, ta, tb, m, n, k, 1.0, dA, lda, dB, ldb, beta, dC, m, -1, stream)
            torch.cuda.synchronize()
            for first in (variants[0], variants[3]):
                G.release_workspace()
                call(*first)
                torch.cuda.synchronize()
                held = G.workspace_info()
                for v in variants:
                    dC.copy_(C0)
                    call(*v)
                    torch.cuda.synchronize()
                    want = dC.clone()
                    graph = torch.cuda.CUDAGraph()
                    with torch.cuda.graph(graph, stream=stream):
                        call(*v)
                    for _ in range(3):
                        dC.copy_(C0)
                        graph.replay()
                        torch.cuda.synchronize()
                        assert torch.equal(dC.view(torch.uint8), want.view(torch.uint8)), (shape, v)
                    assert G.workspace_info() == held, (shape, v)
    G.release_workspace()


@pytest.mark.gpu
def test_reports_time_the_automatic_pick():
    """The report driver and the benchmark main without a config id run MMBO_CONFIG_AUTO and print what it ran."""
    import json
    import sys
    r = subprocess.run([sys.executable, "-m", "gemm_mmbo_amd.report", "shapes", "h,N,N,16,4096,4096", "--reps", "3"], cwd=ROOT,
                       capture_output=True, text=True, timeout=200)
    assert r.returncode == 0, r.stderr[-2000:]
    rec = [json.loads(l) for l in r.stdout.splitlines() if l.startswith("{")][0]
    assert "_WAVE" in rec["config"] and rec["config_id"] == -1 and rec["max_rel_err"] <= U.tol(F16, 4096)
    r = subprocess.run([os.path.join(ROOT, "gemm_mmbo_amd/host/benchmark"), "0", "16", "4096", "4096", "16", "4096", "16", "N", "N", "h", "1", "1", "0"],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "_WAVE" in r.stdout, r.stdout + r.stderr


@pytest.fixture(scope="module")
def asm_files(tmp_path_factory):
    """The generated code of every (element type, tile) the library ships."""
    from concurrent.futures import ThreadPoolExecutor
    outdir = tmp_path_factory.mktemp("wave")

    def compile_one(unit):
        dtype, tile = unit
        out = str(outdir / f"wave_{dtype}_{tile}.s")
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                            "-packed-fp32-ops", "-Wno-unused-command-line-argument", "--cuda-device-only", "-S",
                            f"-DMMBO_DTYPE={dtype}", f"-DMMBO_TILE={tile}", os.path.join(CSRC, "inst_wave.hip"), "-o", out],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        return out
    with ThreadPoolExecutor(max_workers=8) as ex:
        return list(ex.map(compile_one, SHIPPED))


def _lines(path):
    """(inside an asm statement?, instruction or label) of one file."""
    inside = False
    for line in open(path):
        t = line.strip()
        if t.startswith(";;#ASMSTART"):
            inside = True
        elif t.startswith(";;#ASMEND"):
            inside = False
        elif t and (not t.startswith((";", ".")) or t.startswith(".LBB")):
            yield inside, t.split(";")[0].strip()


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_generated_code(asm_files):
    """The direct loads set M0 inside their asm statement without telling the compiler, which must therefore not use M0
    itself; and nothing is spilled (a reload would wait for the direct loads in flight)."""
    for path in asm_files:
        own = [t for inside, t in _lines(path) if not inside]
        assert open(path).read().count(".amdhsa_kernel") == 4, path
        assert not [t for t in own if re.search(r"\bm0\b", t)], path
        assert not [t for t in own if t.startswith("scratch_")], path


def _reads_that_may_overtake(lines):
    """LDS reads that some path reaches from an LDS write without a barrier or an asm wait (which the compiler moves no access
    across) on the way."""
    label = {t[:-1]: i for i, (_, t) in enumerate(lines) if t.endswith(":")}
    bad, seen = set(), set()
    todo = [i + 1 for i, (_, t) in enumerate(lines) if t.startswith("ds_write")]
    while todo:
        i = todo.pop()
        while i < len(lines) and i not in seen:
            seen.add(i)
            inside, t = lines[i]
            if t.startswith(("s_barrier", "s_endpgm")) or (inside and "lgkmcnt(0)" in t):
                break
            if t.startswith("ds_read"):
                bad.add(t)
            if t.startswith(("s_branch", "s_cbranch")):
                todo.append(label[t.split()[-1]])
                if t.startswith("s_branch"):
                    break
            i += 1
    return bad


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_slices_filled_through_registers_are_read_behind_a_wait(asm_files):
    """A partial slice is written to LDS by all lanes and read by other lanes: the reads stay behind the writes only if the
    compiler is told so."""
    planted = [(False, "ds_write_b128 v0, v[1:4]"), (False, "s_waitcnt lgkmcnt(0)"), (False, "ds_read_b128 v[4:7], v0")]
    assert _reads_that_may_overtake(planted) and not _reads_that_may_overtake([planted[0], (True, planted[1][1]), planted[2]])
    for path in asm_files:
        lines = list(_lines(path))
        assert any(t.startswith("ds_write_b128") for _, t in lines)
        assert not _reads_that_may_overtake(lines), path
