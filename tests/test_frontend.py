"""The front-ends of the CPython module (csrc/frontend.cc) beside the Python functions they stand in for: what is accepted, what is refused, and
with which error, form by form.  No call of these reaches a device: they end at a size of zero or at an argument check."""
import inspect

import numpy as np
import pytest

import gemm_mmbo_amd as G
from gemm_mmbo_amd import api


class Tensor:
    def __init__(self, p=64):
        self.p = p

    def data_ptr(self):
        return self.p


class Broken:
    def data_ptr(self):
        raise ValueError("no storage")


class Stream:
    cuda_stream = 0


PLAIN = [0, 0, 0, 0, 5, 6, 1.0, Tensor(), 5, Tensor(), 6, 0.0, Tensor(), 5]
BATCHED = [1, 1, 0, 4, 5, 0, 1.0, 64, 6, 30, None, 6, 30, 0.0, Tensor(), 4, 20, 0]
CHANGES = [{}, {0: 2}, {0: 7}, {0: 2 ** 32 + 2}, {0: True}, {0: "0"}, {1: 2}, {2: -1}, {3: -1}, {3: np.int64(0)}, {3: np.int64(4), 12: None}, {3: 4.0}, {3: 2 ** 70},
           {4: None}, {6: 1}, {6: np.float32(2)}, {6: np.float64(2)}, {6: "x"}, {6: None}, {6: 10 ** 400}, {7: None}, {7: 0}, {7: -8}, {7: Broken(), 3: 4}, {7: object()},
           {7: np.zeros(3)}, {8: 0}, {8: 2 ** 31}, {3: 4, 12: None}, {3: 4, 7: None}, {3: 4, 9: None}]
TAILS = [(), (-1,), (10 ** 6,), (-2,), (None,), (-1, None), (-1, 0), (-1, Stream()), (-1, object()), (-1, None, 3)]


def _result(f, args, kw):
    try:
        return f(*args, **kw)
    except Exception as e:                       # (what it is and what it says)
        return type(e), str(e)


@pytest.mark.skipif(api._frontend is None, reason="the module is not built")
@pytest.mark.parametrize("which", [0, 1, 2])
def test_every_form_of_a_call_gives_what_the_python_function_gives(which):
    ours = (G.gemm, G.gemm_strided_batched, G.gemm_strided_batched_static_workspace)[which]
    python = api._PYTHON_FRONT_ENDS[which]
    assert ours is not python and inspect.signature(ours) == inspect.signature(python) and ours.__name__ == python.__name__
    base, taken = (PLAIN if which == 0 else BATCHED), set()
    names = list(inspect.signature(python).parameters)
    for change in CHANGES:
        for tail in TAILS:
            args = list(base)
            for i, v in change.items():
                args[i] = v
            full = args + list(tail)
            forms = [(full, {})] + [(full[:cut], dict(zip(names[cut:], full[cut:]))) for cut in (3, 0) if len(full) <= len(names)]
            for a, kw in forms + [(args[:-1], {})]:
                got, want = _result(ours, a, kw), _result(python, a, kw)
                assert got == want, (a, kw, got, want)
                taken.add(want if want is None else want[0])
    assert {None, G.MmboError, TypeError} <= taken


@pytest.mark.skipif(api._frontend is None, reason="the module is not built")
def test_arguments_are_not_kept():
    import sys
    t = Tensor()
    before = sys.getrefcount(t)
    for _ in range(50):
        G.gemm(0, 0, 0, 0, 5, 6, 1.0, t, 5, t, 6, 0.0, t, 5)
        with pytest.raises(G.MmboError):
            G.gemm(0, 0, 0, 4, 5, 6, 1.0, t, 0, t, 6, 0.0, t, 5)
    assert sys.getrefcount(t) == before
