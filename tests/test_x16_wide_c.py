"""The 16x16-block ring kernel's element-wise epilogue, for a C whose tiles span more than the 32-bit offsets of a buffer access, on
ragged problems: the shifted rows and columns of either operand, cut groups, a partial last slice, odd leading dimensions."""
import pytest

import util as U

F32, F16 = U.F32, U.F16
NAMES = {F32: "f32", F16: "f16"}
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,ldc", [(F32, (1 << 21) + 64), (F16, (1 << 22) + 67)], ids=["f32", "f16"])
def test_ragged_c_whose_tile_span_passes_32_bit_offsets(dtype, ldc):
    import torch

    import gemm_mmbo_amd as G
    m, n, k = 256 + 3, 256 + 1, 70
    t = torch.float32 if dtype == F32 else torch.float16
    cid = next(c for c in range(G.num_configs(dtype)) if "_ACC" in (d := G.config_info(dtype, c))["name"] and d["split_k"] == 1 and
               d["macro_tile_m"] == d["macro_tile_n"] == 256)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    C = torch.zeros(ldc * n, device="cuda", dtype=t)
    Cv = C.view(n, ldc)
    for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
        A, B = ((torch.rand(count, device="cuda", generator=gen) * 2 - 1).to(t) for count in (m * k, k * n))
        a = (A.view(m, k).t() if ta else A.view(k, m)).double().contiguous()           # k x m, as column-major C is the transpose
        b = (B.view(k, n).t() if tb else B.view(n, k)).double().contiguous()           # n x k
        for beta in (0.0, 0.5):
            C0 = (torch.rand(n, m, device="cuda", generator=gen) * 2 - 1).to(t)
            Cv[:, :m] = C0 if beta else float("nan")
            Cv[:, m:m + 16] = 7.0                                                     # sentinels right below the window
            G.gemm(dtype, ta, tb, m, n, k, -1.5, A, k if ta else m, B, n if tb else k, beta, C, ldc, cid)
            torch.cuda.synchronize()
            want = -1.5 * (b @ a) + (beta * C0.double() if beta else 0.0)
            # fp32 accumulation of k products and the two scalars, each rounding at most 2^-24 of what is added up; fp16 results are
            # rounded once more, to 11 bits (or to the spacing of its subnormals)
            limit = (k + 3) * 2.0 ** -24 * (1.5 * (b.abs() @ a.abs()) + beta * C0.double().abs())
            if dtype == F16:
                limit = limit * (1 + 2.0 ** -10) + 2.0 ** -11 * want.abs() + 2.0 ** -25
            bad = (Cv[:, :m].double() - want).abs() > limit
            assert not bool(bad.any()) and not bool(Cv[:, :m].isnan().any()), f"{NAMES[dtype]} {'NT'[ta]}{'NT'[tb]} beta {beta}: {int(bad.sum())}"
            assert bool((Cv[:, m:m + 16] == 7.0).all()) and float(Cv[:, m + 16:].abs().max()) == 0.0
    del C, Cv
    torch.cuda.empty_cache()
