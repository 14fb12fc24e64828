"""16-bit products of a deep K: 256x256 tiles whose depth is dealt to workgroups, whole and ragged at
both edges, and 128x128 instead of 64x128 tiles from a depth of 2048 on.  Against the product in
float64, element by element, within the rounding of K fp32 additions (the products are exact)."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, _name, cases

SPLIT = "K dealt to 4 workgroups per tile"
FORMS = [((2048, 2048, 16384, "bfloat16", "nt"), "256x256x32", SPLIT), ((1960, 2040, 16384, "bfloat16", "nn"), "256x256x32", SPLIT),
         ((2000, 1928, 16512, "float16", "tn"), "256x256x32", "K dealt to 4"), ((4096, 1024, 8192, "bfloat16", "nn"), "128x256x32", "K dealt to 2"),
         ((1550, 2000, 2048, "bfloat16", "nt"), "128x128x64", ""), ((1552, 2000, 2112, "float16", "tn"), "128x128x64", ""), ((1550, 2000, 1984, "bfloat16", "nt"), "64x128x64", "")]


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c,tile,split", FORMS, ids=lambda v: _name(v) if isinstance(v, tuple) else "")
def test_stays_in_bounds(c, tile, split, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    desc = _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert tile in desc and split in desc and (split or "K dealt" not in desc)
    assert hostcheck.check_schedule(hiplib, pf.schedule, max_threads=1 << 14) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c,tile,split", FORMS, ids=lambda v: _name(v) if isinstance(v, tuple) else "")
def test_against_float64(c, tile, split):
    m, n, k, dtype, layout = c
    state = cases.prepare(_case(*c), 5)
    desc = state["plan"].kernel_info()[0]["desc"]
    assert tile in desc and split in desc
    got = cases.run(state)["C"]
    state["plan"].sync()
    by = {s.name: state["data"][s.index].double() for s in state["plan"].external_slots()}
    a = by["A"].reshape(k, m).T if layout[0] == "t" else by["A"].reshape(m, k)
    b = by["B"].reshape(n, k).T if layout[1] == "t" else by["B"].reshape(k, n)
    err = (got.double().reshape(m, n) - a @ b).abs()
    bound = k * 2.0 ** -24 * (a.abs() @ b.abs())
    assert bool((err <= bound).all()), float((err / bound).max())
