"""Where the automatic pick takes fp32 products in bf16 planes (gemm_planes.hpp): never in sums of so much longer runs of k that they are less exact
than those of the fp32 matrix instructions, whose runs the cases name."""
import re

import numpy as np
import pytest

import util as U

F32 = U.F32


def _runs(info):
    lsu = re.search(r"LSU(\d+)", info["name"])
    return info["split_k"] * (int(lsu.group(1)) if lsu else 1)


@pytest.mark.parametrize("ta,tb,m,n,k,batch,others", [
    (1, 1, 384, 384, 2048, 16, 4), (1, 0, 96, 384, 32768, 64, 8), (0, 1, 640, 512, 16384, 4, 4), (1, 0, 300, 300, 20000, 1, 32), (0, 0, 128, 5120, 8192, 1, 8),
    (1, 1, 704, 719, 25984, 1, 16), (0, 1, 568, 62, 49646, 1, 64), (1, 1, 288, 288, 26240, 1, 64), (1, 0, 2080, 1024, 2176, 1, 4),
    (0, 1, 4264, 256, 256, 1, 4), (0, 0, 858, 1408, 768, 1, 4),
])
def test_runs_in_planes_are_not_too_long(ta, tb, m, n, k, batch, others):
    import gemm_mmbo_amd as G
    info = G.auto_info(F32, ta, tb, m, n, k, batch)
    if "_BF16X3" in info["name"]:
        assert k // others >= 128 and _runs(info) * (1 if k // others < 256 else 2 if k <= 4096 else 1.5) >= others, info["name"]


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb,m,n,k,batch,others", [
    (1, 1, 384, 384, 2048, 16, ("MT192x192", "_MFMA16x16x4_ACC", 4)), (0, 0, 128, 5120, 8192, 1, ("MT064x064", "_RING6", 8)),
    (0, 1, 640, 512, 16384, 4, ("MT064x064", "_RING6", 4)),
])
def test_the_pick_is_as_exact_as_the_fp32_matrix_instructions_it_replaces(ta, tb, m, n, k, batch, others):
    """2-norm of the error against 64 bits on the same operands.  By 3 %: where runs in planes may be twice as long, the two are equal on the widest
    spread of operands, and two sets of a million roundings give it to about 1 %."""
    import gemm_mmbo_amd as G
    tile, family, split = others
    native = next(c for c in range(G.num_configs(F32)) if (d := G.config_info(F32, c))["name"].startswith(tile) and d["name"].endswith(family) and d["split_k"] == split)
    for dist in ("uniform", "positive", "spread"):
        p = U.Problem(F32, ta, tb, m, n, k, batch=batch, seed=k)
        if dist == "positive":
            p.A, p.B = np.abs(p.A), np.abs(p.B)
        if dist == "spread":
            rng = np.random.default_rng(k)
            p.A = (p.A * np.exp2(rng.uniform(-20, 20, p.A.size))).astype(np.float32)
            p.B = (p.B * np.exp2(rng.uniform(-20, 20, p.B.size))).astype(np.float32)
        a, b = (x.reshape((batch, -1, ld)).astype(np.float64) for x, ld in ((p.A, p.lda), (p.B, p.ldb)))
        want = ((b if not tb else b.transpose(0, 2, 1)) @ (a if not ta else a.transpose(0, 2, 1))).reshape(-1)      # (C's columns, one after the other)

        def error(got):
            return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))
        here, limit = error(U.run_gpu(p)[0]), error(U.run_gpu(p, native)[0])
        assert here <= 1.03 * limit, (dist, here, limit)


@pytest.mark.parametrize("ta,tb,m,n,k,batch,name,split", [
    (0, 1, 5120, 5120, 1024, 1, "MT256x128x32", 1), (0, 1, 44160, 2048, 256, 1, "MT256x128x32", 1), (1, 0, 2500, 1500, 700, 1, "MT128x128x32", 1),
    (0, 0, 256, 256, 256, 64, "MT128x128x32", 1), (1, 0, 640, 384, 10000, 1, "MT128x064x32", 8), (0, 1, 768, 768, 2048, 3, "MT128x064x32", 1),
    (0, 0, 1024, 1024, 1024, 1, "MT064x064x32", 1), (1, 1, 800, 900, 1300, 1, "MT064x064x32", 1),
])
def test_the_pick_reaches_every_tile(ta, tb, m, n, k, batch, name, split):
    import gemm_mmbo_amd as G
    info = G.auto_info(F32, ta, tb, m, n, k, batch)
    assert info["name"].startswith(name) and "_BF16X3" in info["name"] and info["split_k"] == split, info["name"]
    # k is split over work-groups only where the tables' pick needs a workspace, too
    assert split == 1 or G.config_info(F32, G.select_config(F32, ta, tb, m, n, k, batch))["split_k"] > 1


@pytest.mark.parametrize("dtype,ta,tb,m,n,k,batch,ld", [
    (U.F32, 0, 0, 512, 512, 512, 1, {}),                        # a few microseconds
    (U.F32, 0, 0, 3, 9000, 8192, 1, {}), (U.F32, 1, 1, 9000, 3, 8192, 1, {}),       # less than 16 bytes of a contiguous dimension
    (U.F32, 0, 0, 4096, 4096, 63, 1, {}), (U.F32, 0, 0, 4096, 4096, 0, 1, {}),
    (U.F32, 1, 0, 5000, 5000, 5000, 1, {"lda": 1 << 23}),       # 128 rows and more span 2 GiB
    (U.F16, 0, 0, 4096, 4096, 4096, 1, {}), (U.F64, 0, 0, 4096, 4096, 4096, 1, {}),
])
def test_where_the_pick_does_not_take_planes(dtype, ta, tb, m, n, k, batch, ld):
    import gemm_mmbo_amd as G
    assert "BF16X3" not in G.auto_info(dtype, ta, tb, m, n, k, batch, **ld)["name"]


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb,m,n,k,batch,split,tile", [(1, 1, 3000, 1500, 6144, 1, 1, 1), (0, 0, 256, 1500, 16384, 2, 8, 1), (1, 0, 2304, 768, 6144, 3, 1, 0)])
def test_partial_sums_that_the_static_workspace_does_not_hold(ta, tb, m, n, k, batch, split, tile):
    """The entry point that allocates nothing runs the same tile with the largest split whose partial sums fit: bit for bit what that split gives."""
    import torch

    import gemm_mmbo_amd as G
    import test_planes_kernel as P
    info = G.auto_info(F32, ta, tb, m, n, k, batch)
    assert info["name"].startswith("MT%03dx%03dx32" % P.TILES[tile]) and "_BF16X3" in info["name"]
    sums = m * n * batch * 4
    assert info["split_k"] * sums > G.static_workspace_bytes() >= split * sums * (split > 1) and 2 * split * sums > G.static_workspace_bytes()
    p = U.Problem(F32, ta, tb, m, n, k, batch=batch, seed=split)
    A, B, C = (torch.from_numpy(x).cuda() for x in (p.A, p.B, p.C))
    G.gemm_strided_batched_static_workspace(F32, ta, tb, m, n, k, 1.0, A, p.lda, p.sa, B, p.ldb, p.sb, 0.0, C, p.ldc, p.sc, batch)
    torch.cuda.synchronize()
    assert np.array_equal(C.cpu().numpy(), P._run(p, tile, split)[0])


CHANGES = [(1, 1, 4373, 72, 15807), (0, 0, 7440, 41, 14752)]


def _calls(ta, tb, m, n, k):
    """(padding of the leading dimensions, beta): calls of one shape that go to planes, and to another kernel whose runs planes would lengthen."""
    import gemm_mmbo_amd as G
    calls = [(0, 0.0), (1, 0.5), (0, 0.5)]
    return calls, [G.auto_info(F32, ta, tb, m, n, k, 1, (k if ta else m) + pad, (n if tb else k) + pad, m, beta != 0)["name"] for pad, beta in calls]


@pytest.mark.parametrize("shape", CHANGES)
def test_calls_of_one_shape_may_differ_in_the_kernel(shape):
    names = _calls(*shape)[1]
    assert "_BF16X3" in names[0] and "_BF16X3" not in names[1], names


@pytest.mark.gpu
@pytest.mark.parametrize("shape", CHANGES)
def test_one_call_of_such_a_shape_leaves_the_workspace_of_all(shape):
    """Either kind of call first, then each captured: nothing is allocated, and each replay gives the bits of the eager call."""
    import torch

    import gemm_mmbo_amd as G
    ta, tb, m, n, k = shape
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        A, B, C0 = (torch.rand(x, device="cuda") for x in ((m + k + 1) + (m + 1) * (k + 1), (n + k + 1) + (n + 1) * (k + 1), m * n))
        C = C0.clone()

        def call(pad, beta):
            G.gemm(F32, ta, tb, m, n, k, 1.0, A, (k if ta else m) + pad, B, (n if tb else k) + pad, beta, C, m, -1, stream)
        calls = _calls(*shape)[0]
        for first in calls[:2]:
            torch.cuda.synchronize()
            G.release_workspace()
            call(*first)
            torch.cuda.synchronize()
            held = G.workspace_info()
            for c in calls:
                C.copy_(C0)
                call(*c)
                torch.cuda.synchronize()
                want = C.clone()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=stream):
                    call(*c)
                for _ in range(3):
                    C.copy_(C0)
                    graph.replay()
                    torch.cuda.synchronize()
                    assert torch.equal(C, want), (shape, c)
                assert G.workspace_info() == held, (shape, c)
    G.release_workspace()
