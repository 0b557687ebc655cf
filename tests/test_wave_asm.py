"""The split-by-wavefront kernel's partial last slice, on the gfx950 assembly hipcc generates (no GPU needed): lines and groups that do
not exist are left to the range check of buffer loads.  Plain loads, which repeat the last line instead, cost every ragged k."""
import os

import pytest

import test_kernel_asm as K

pytestmark = pytest.mark.skipif(not os.path.exists(K.HIPCC), reason="hipcc not installed")


def test_partial_slices_request_only_what_exists(tmp_path):
    path = K._compile(("inst_wave.hip", ["-DMMBO_DTYPE=1", "-DMMBO_TILE=1"]), str(tmp_path))
    kernels = {name: body for name, body in K._kernels(path).items() if any(t.startswith("v_mfma") for t in body)}
    assert len(kernels) >= 4
    for name, body in kernels.items():
        # (fp16: the old C comes in 8-byte groups, an operand shorter than 16 bytes by elements)
        assert not [t for t in body if t.startswith("global_load_dwordx4")], name
        assert [t for t in body if t.startswith("buffer_load_dwordx4") and "lds" not in t], name
