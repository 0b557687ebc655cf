"""What the fp64 kernel's speed rests on in the generated code (no GPU needed): in the loop over whole stages the operands of the
next stage go from registers to LDS under the MFMAs of this one, so nothing between the loads and the LDS stores may depend
on the tile, and part of the stage's MFMAs must be left when the stores are issued; the loads of a partial stage are in flight
together."""
import os
import subprocess

import pytest

import test_kernel_asm as K

pytestmark = pytest.mark.skipif(not os.path.exists(K.HIPCC), reason="hipcc not installed")


def _whole_stage_loops(body):
    """Innermost loops that load, multiply and store to LDS, each as its list of instructions from label to back edge."""
    label, loops = {}, []
    for i, t in enumerate(body):
        if t.endswith(":"):
            label[t[:-1]] = i
        elif t.startswith(("s_cbranch", "s_branch")) and t.split()[-1] in label:
            loops.append((label[t.split()[-1]], i))
    inner = [(a, b) for a, b in loops if not any(a <= c and d < b for c, d in loops)]
    out = []
    for a, b in inner:
        loop = [t for t in body[a:b + 1] if not t.endswith(":")]
        if all(any(t.startswith(p) for t in loop) for p in ("global_load_dwordx4", "v_mfma_f64", "ds_write", "s_barrier")):
            out.append(loop)
    return out


def _stores_after_every_mfma(loop):
    """The loop as a cycle from its first load on: is the last MFMA issued before the first LDS store?"""
    first_load = next(i for i, t in enumerate(loop) if t.startswith("global_load"))
    turn = loop[first_load:] + loop[:first_load]
    mfma = [i for i, t in enumerate(turn) if t.startswith("v_mfma")]
    store = next(i for i, t in enumerate(turn) if t.startswith("ds_write"))
    return mfma[-1] < store


# 8-byte loads a thread makes for a partial stage of both operands: rows x 16 of k / threads, for each row of the config table
PARTIAL_LOADS = [(128 + 128) * 16 // 256, (256 + 128) * 16 // 512, (64 + 64) * 16 // 256, (32 + 32) * 16 // 256, (128 + 128) * 16 // 512,
                 (128 + 64) * 16 // 256]


def _most_8_byte_loads_in_flight(body):
    """The longest run of 8-byte loads without a wait for loads, a branch or a label among them."""
    most = run = 0
    for t in body:
        if t.startswith("global_load_dwordx2"):
            run += 1
            most = max(most, run)
        elif t.endswith(":") or t.startswith(("s_cbranch", "s_branch")) or (t.startswith("s_waitcnt") and "vmcnt" in t):
            run = 0
    return most


def test_loop_finder_on_planted_code():
    loop = [".LBB0_1:", "global_load_dwordx4 v[0:3], v4, s[0:1]", "v_mfma_f64_16x16x4_f64 a", "ds_write_b128 v9, v[0:3]",
            "v_mfma_f64_16x16x4_f64 b", "s_barrier", "s_cbranch_scc1 .LBB0_1"]
    assert _whole_stage_loops(["s_nop 0"] + loop) == [loop[1:]]
    assert not _stores_after_every_mfma(loop[1:])
    late = loop[1:3] + [loop[4], "v_cndmask_b32_e32 v0, v0, v2, vcc", loop[3]] + loop[5:]
    assert _stores_after_every_mfma(late)


@pytest.mark.parametrize("tile", range(6))
def test_lds_stores_run_under_the_mfmas(tile, tmp_path):
    out = str(tmp_path / "dgemm.s")
    r = subprocess.run([K.HIPCC] + K.FLAGS + [f"-DMMBO_TILE={tile}", os.path.join(K.CSRC, "inst_dgemm.hip"), "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = K._kernels(out)
    assert len(kernels) in (4, 8)
    for name, body in kernels.items():
        loops = _whole_stage_loops(body)
        assert loops, name
        for loop in loops:
            assert not [t for t in loop if t.startswith(("v_cndmask", "scratch_"))], name
            assert not _stores_after_every_mfma(loop), name
        assert _most_8_byte_loads_in_flight(body) >= PARTIAL_LOADS[tile], name
