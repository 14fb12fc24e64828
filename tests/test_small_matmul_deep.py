"""Deep 16-bit products of few tiles on the template whose waves share the depth: 16x16 tiles where each has a CU, 32x32
where 16x32 tiles would share them, on both sides of either line, ragged rows, columns and depths, every layout.  Against the
product in float64, element by element, within the rounding of K fp32 additions (the products are exact)."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, _name, cases

FORMS = [((12, 768, 3072, "bfloat16", "nn"), "16x16"), ((64, 512, 4096, "bfloat16", "nt"), "16x16"), ((49, 610, 2050, "float16", "tn"), "16x16"),
         ((64, 1024, 2048, "bfloat16", "nn"), "16x16"), ((64, 1030, 2048, "bfloat16", "nn"), "16x32"), ((64, 512, 2046, "bfloat16", "nt"), "16x32"),
         ((300, 500, 1028, "bfloat16", "nn"), "32x32"), ((290, 514, 1500, "float16", "tn"), "32x32"), ((257, 482, 1030, "bfloat16", "nt"), "32x32"),
         ((256, 512, 1028, "bfloat16", "nn"), "16x32"), ((300, 500, 1022, "bfloat16", "nn"), "16x32")]


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c,tile", FORMS, ids=lambda v: _name(v) if isinstance(v, tuple) else v)
def test_stays_in_bounds(c, tile, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert f"tile {tile}, depth dealt to 8 waves" in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c,tile", FORMS, ids=lambda v: _name(v) if isinstance(v, tuple) else v)
def test_against_float64(c, tile):
    m, n, k, dtype, layout = c
    state = cases.prepare(_case(*c), 6)
    assert f"tile {tile}, depth dealt to 8 waves" in state["plan"].kernel_info()[0]["desc"]
    got = cases.run(state)["C"]
    state["plan"].sync()
    by = {s.name: state["data"][s.index].double() for s in state["plan"].external_slots()}
    a = by["A"].reshape(k, m).T if layout[0] == "t" else by["A"].reshape(m, k)
    b = by["B"].reshape(n, k).T if layout[1] == "t" else by["B"].reshape(k, n)
    err = (got.double().reshape(m, n) - a @ b).abs()
    assert bool((err <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all())
