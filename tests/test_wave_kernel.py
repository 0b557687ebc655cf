"""The split-by-wavefront kernel (csrc/gemm_wave.hpp), which the automatic pick takes for small, thin and long-k problems.

GPU: shapes at the edges of its tiles (16, 32, 64 rows), of its slices (32 halves, 16 floats, 8 doubles; pairs of them;
fewer slices than wavefronts), with row-contiguous operands that end inside a 16-byte group or are shorter than one, and
with k long enough for GlobalSplitU beyond 16 (several threads then share the splits of one sum), against the fp64 oracle
with the suite's own bounds.  CPU: facts about the generated code that the kernel's asm statements rely on.
"""
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
    for i, (m, n, k, batch) in enumerate(SHAPES):
        pad = (0, 1, 8)[i % 3]
        ar, br = U.stored_shape(ta, m, k)[0], U.stored_shape(tb, k, n)[0]
        p = U.Problem(dtype, ta, tb, m, n, k, -1.5, (0.0, 0.5)[i % 2], lda=ar + pad, ldb=br + pad, ldc=m + pad, batch=batch,
                      seed=300 + i, dist="normal" if dtype == F16 else "uniform", c_fill=("nan", "uniform")[i % 2])
        got, guard = U.run_gpu(p)
        U.check(p, got, f"{NAMES[dtype]} {'NT'[ta]}{'NT'[tb]} {m}x{n}x{k} b{batch}")
        assert np.all(guard == 0)
        # the entry point that allocates nothing: the same bits
        dA, dB, dC = (torch.from_numpy(x).cuda() for x in (p.A, p.B, p.C))
        G.gemm_strided_batched_static_workspace(dtype, ta, tb, m, n, k, -1.5, dA, p.lda, p.sa, dB, p.ldb, p.sb, p.beta, dC, p.ldc,
                                                p.sc, batch)
        torch.cuda.synchronize()
        assert np.array_equal(dC.cpu().numpy().view(U.BITS[dtype]), got.view(U.BITS[dtype]))


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


NUM_TILES = 8


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
        return list(ex.map(compile_one, [(d, t) for d in (0, 1, 2) for t in range(NUM_TILES)]))


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
