"""The build where the CPython module of the front-ends cannot be built: the library is there all the same, and no older module beside it."""
import os

import pytest

from gemm_mmbo_amd import build as B


@pytest.mark.parametrize("compiler", ["/nonexistent/g++", "false"])
def test_the_library_is_built_without_the_module(tmp_path, monkeypatch, capsys, compiler):
    objects = [os.path.join(B.OBJ, u[1]) for u in B._units()]
    if not os.path.exists(B.HIPCC) or not all(os.path.exists(o) for o in objects):
        pytest.skip("needs hipcc and built objects")
    old = tmp_path / "_frontend.so"
    old.write_bytes(b"of older sources")
    os.utime(old, (0, 0))
    monkeypatch.setattr(B, "FRONTEND", str(old))
    monkeypatch.setattr(B, "LIB", str(tmp_path / "lib.so"))
    monkeypatch.setattr(B, "_compile", lambda unit, force, newest: (unit[1], "up to date"))
    monkeypatch.setenv("CXX", compiler)
    assert os.path.exists(B.build(verbose=False))
    assert not old.exists()
    assert "was not built" in capsys.readouterr().err
