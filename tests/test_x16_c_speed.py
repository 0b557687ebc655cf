"""Where the columns of a C that is updated or written start must not decide what a call costs: the time of the 16x16-block ring
kernel on columns at any element, against the time of the same call on columns that it has always served well."""
import pytest

import util as U

pytestmark = pytest.mark.gpu


def _times(m, n, k, ta, tb, beta, forms, reps, rounds=15):
    """Median time of a call for every (ldc, offset of C in elements), fp16, the forms in turn."""
    import torch

    import gemm_mmbo_amd as G
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    A, B = ((torch.randn(m * k if i == 0 else k * n, device="cuda", generator=gen) * 0.1).half() for i in range(2))
    C = torch.zeros(max(ldc for ldc, _ in forms) * n + 16, device="cuda", dtype=torch.float16)
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    times = [[] for _ in forms]
    for r in range(rounds + 1):
        for i, (ldc, offset) in enumerate(forms):
            start.record()
            for _ in range(reps):
                G.gemm(U.F16, ta, tb, m, n, k, 1.0, A, k if ta else m, B, n if tb else k, beta, C.data_ptr() + 2 * offset, ldc)
            end.record()
            end.synchronize()
            if r > 0:
                times[i].append(start.elapsed_time(end) / reps)
    return [sorted(t)[len(t) // 2] for t in times]


@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_odd_columns_cost_the_same_whatever_element_c_starts_on(beta):
    """16-byte accesses off a dword boundary took 1.25 to 1.5 times as long as the epilogue for odd columns."""
    known, all_odd, half_odd = _times(8192, 2048, 256, 0, 1, beta, [(8193, 0), (8192, 1), (8193, 1)], 100)
    assert all_odd <= 1.15 * known and half_odd <= 1.15 * known, (known, all_odd, half_odd)


def test_large_product_into_columns_off_16_bytes():
    """With the streaming hint, whose stores of partial lines nothing merges: 1.13 times the time of whole lines."""
    aligned, off = _times(8192, 8192, 4096, 0, 0, 0.0, [(8192, 0), (8192, 2)], 6)
    assert off <= 1.07 * aligned, (aligned, off)
