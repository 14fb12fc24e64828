"""16-bit products of more rows than whole rounds of 256x256 tiles take: the rows left over go to a launch of 64x128
tiles of their own.  Ragged edges of both, every layout.  Against the product in float64, element by element,
within the rounding of K fp32 additions (K * 2^-24 * sum of |a b|; the products of 16-bit values are exact)."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SHAPES = [(49452, 1000, 512, "bfloat16", "nn"), (49217, 1001, 1600, "float16", "nt"), (49224, 1024, 512, "bfloat16", "tn")]


def _case(m, n, k, dtype, layout):
    return dict(kind="matmul", m=m, n=n, k=k, dtype=dtype, layout=layout)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_stays_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert "rows from 49152 on by a launch of 64x128 tiles" in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert hostcheck.check_schedule(hiplib, pf.schedule, max_threads=1 << 14) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_against_float64(c):
    m, n, k, dtype, layout = c
    state = cases.prepare(_case(*c), 5)
    assert "rows from 49152 on" in state["plan"].kernel_info()[0]["desc"]
    got = cases.run(state)["C"]
    state["plan"].sync()
    by = {s.name: state["data"][s.index].double() for s in state["plan"].external_slots()}
    a = by["A"].reshape(k, m).T if layout[0] == "t" else by["A"].reshape(m, k)
    b = by["B"].reshape(n, k).T if layout[1] == "t" else by["B"].reshape(k, n)
    err = (got.double().reshape(m, n) - a @ b).abs()
    assert bool((err <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all())
