"""Products whose operands are written as 16-bit planes first (kernels/operand_split.hip), both
by one launch: extents at, below and above the edges of its 64x64 tiles, rows that are and are
no multiple of 8 long, every layout, bf16 and fp16 operands, more tiles for one operand than
for the other.  Against the product in float64, element by element, within the rounding of K
fp32 additions (K * 2^-24 * sum of |a b|; the products of 16-bit values are exact)."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, _name, cases

PLANES = [(129, 66, 131, "bfloat16", "nn"), (64, 193, 127, "float16", "nt"), (128, 71, 129, "float16", "nn"), (257, 65, 72, "bfloat16", "tn"),
          (65, 130, 200, "float16", "nt"), (191, 67, 130, "float16", "tn"), (70, 700, 1001, "bfloat16", "nt"), (1111, 999, 1501, "float16", "nn")]
FORMS = dict(bfloat16="written as bf16 planes first (1 + 1 planes", float16="written as fp16 planes first (1 + 1 planes")


@pytest.fixture
def planes(monkeypatch):
    monkeypatch.setenv("POLY_HIP_BF16_SPLIT_MIN", "1")
    monkeypatch.setenv("POLY_HIP_NO_WAVE_MM", "1")


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", PLANES, ids=_name)
def test_stays_in_bounds(c, hiplib, monkeypatch, planes):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert FORMS[c[3]] in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c", PLANES, ids=_name)
def test_against_float64(c, planes):
    m, n, k, dtype, layout = c
    state = cases.prepare(_case(*c), 6)
    assert FORMS[dtype] in state["plan"].kernel_info()[0]["desc"]
    got = cases.run(state)["C"]
    state["plan"].sync()
    by_name = {s.name: state["data"][s.index] for s in state["plan"].external_slots()}
    a, b = by_name["A"].double().cpu(), by_name["B"].double().cpu()
    a = a.reshape(k, m).T if layout[0] == "t" else a.reshape(m, k)
    b = b.reshape(n, k).T if layout[1] == "t" else b.reshape(k, n)
    err = (got.double().cpu().reshape(m, n) - a @ b).abs()
    bound = k * 2.0 ** -24 * (a.abs() @ b.abs())
    assert bool((err <= bound).all()), float((err / bound).max())
