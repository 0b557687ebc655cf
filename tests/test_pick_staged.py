"""Where the automatic pick leaves the kernels of the tables for the split-by-wavefront one, and where it stays (no GPU needed)."""
import pytest

import util as U


@pytest.mark.parametrize("dtype,ta,tb,m,n,k,batch,wave", [
    (U.F16, 0, 1, 102, 32, 512, 191, True),        # a batch of narrow problems, columns off 16 bytes
    (U.F16, 0, 1, 2, 2267, 7424, 1, True),         # less than 16 bytes of m in memory
    (U.F16, 1, 1, 12320, 4, 5569, 1, True),
    (U.F32, 0, 1, 3, 9000, 4096, 1, True),
    (U.F16, 1, 1, 37, 384, 397, 229, False),       # over 32 wide, a wavefront per work-group
    (U.F32, 1, 0, 56, 512, 384, 128, False),
    (U.F64, 0, 0, 736, 256, 17856, 1, True),       # a work-group's slices at a round trip each
    (U.F64, 0, 1, 44160, 2048, 384, 1, False),
    (U.F64, 0, 0, 2048, 2048, 2048, 1, False),
    (U.F16, 0, 0, 32, 32, 32, 1, None),            # a few microseconds: either
])
def test_where_the_pick_leaves_the_tables(dtype, ta, tb, m, n, k, batch, wave):
    import gemm_mmbo_amd as G
    a = G.auto_info(dtype, ta, tb, m, n, k, batch)
    if wave is None:
        assert a["config_id"] == G.CONFIG_AUTO or a["config_id"] == G.select_config(dtype, ta, tb, m, n, k, batch)
        return
    assert ("WAVE" in a["name"]) == wave, a["name"]
    # whether a call needs a workspace still follows from the pick of the tables
    if a["split_k"] > 1:
        assert G.config_info(dtype, G.select_config(dtype, ta, tb, m, n, k, batch))["split_k"] > 1


@pytest.mark.parametrize("ta,tb,m,n,k,runs", [(1, 1, 55, 4480, 2298, 8), (1, 0, 3232, 36, 3968, 8), (1, 0, 1456, 42, 8064, 16)])
def test_fp32_sums_are_not_added_up_in_fewer_runs_than_the_staged_kernels(ta, tb, m, n, k, runs):
    import re

    import gemm_mmbo_amd as G
    assert "DTL1" not in (staged := G.config_info(U.F32, G.select_config(U.F32, ta, tb, m, n, k)))["name"] and staged["split_k"] == runs
    a = G.auto_info(U.F32, ta, tb, m, n, k)
    lsu = re.search(r"LSU(\d+)", a["name"])
    if "_BF16X3" in a["name"]:                   # (a rule of its own)
        return
    assert a["split_k"] * (int(lsu[1]) if lsu else 1) >= runs, a["name"]
