"""Row chains whose last phase takes a computed row and the operand it came from, both kept (the
shape of a cross-entropy's gradient): the longest rows that stay out of LDS, the shortest and
longest that are partly there, as single elements and as 16-byte vectors; a row that is the only one,
whose operand's positions depend on no row.  Against float64."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SIZES = [(3, 40961, False), (2, 46079, False), (3, 46081, True), (2, 46084, True), (5, 50257, True), (2, 53247, True), (300, 53248, True),
         (1, 20000, False), (1, 40000, False), (1, 50257, True), (1, 53248, True)]


def _plan(rows, cols):
    """out = softmax(x) + 3/4 x, by rows"""
    s = cases.Schedule()
    out, x = s.buf("out", rows * cols), s.buf("x", rows * cols)
    (r,) = s.ranges(rows)
    k = s.rrange(cols)
    mx = s.store(s.tmp(rows), r, s.reduce("MAX", x[r * cols + k], k), r)
    r, k = s.ranges(rows, cols)
    i = r * cols + k
    mid = s.store(s.tmp(rows * cols), i, ((x[i] - mx[r]) * cases.LOG2E).un("EXP2"), r, k)
    (r,) = s.ranges(rows)
    k = s.rrange(cols)
    sm = s.store(s.tmp(rows), r, s.reduce("ADD", mid[r * cols + k], k), r)
    (i,) = s.ranges(rows * cols)
    s.store(out, i, mid[i] / sm[i // cols] + x[i] * 0.75, i)
    return s.plan()


def _source(lib, pf):
    assert lib.poly_hip_fused_groups(pf.schedule, -1, None, None) == 1
    src, n_items = C.c_void_p(), C.c_int()
    lib.poly_hip_fused_groups(pf.schedule, 0, C.byref(src), C.byref(n_items))
    assert n_items.value == 4
    return _ffi.take_string(src.value).split("\n// ---- ")[0]


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("rows,cols,in_lds", SIZES)
def test_in_bounds(rows, cols, in_lds, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _plan(rows, cols)
    text = _source(hiplib, pf)
    assert ("poly_row_kept" in text) == in_lds
    assert "(c0[it] = " in text and text.count("c0[it]") >= 2      # read in the first phase, taken in a later one
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    slots, launch = (C.c_int * 64)(), (C.c_int * 4)()
    n = hiplib.poly_hip_fused_group_launch(pf.schedule, 0, slots, 64, launch)
    sizes = [int(s.buf_slots[slots[i]].nbytes) for i in range(n)]
    hostcheck.check_kernel(text, "poly_k", tuple(launch[:3]), launch[3], sizes, block_stride=max(1, launch[0] * launch[3] >> 16))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,in_lds", SIZES)
def test_against_float64(rows, cols, in_lds):
    import torch
    plan = _plan(rows, cols)
    assert ("in LDS" in plan.kernel_info()[0]["desc"]) == in_lds
    gen = torch.Generator(device="cuda").manual_seed(rows * cols)
    x = torch.randn(rows * cols, device="cuda", generator=gen)
    out = torch.empty_like(x)
    data = [None] * len(plan.slots)
    for s in plan.external_slots():
        data[s.index] = {"x": x, "out": out}[s.name]
    plan.run(data)
    plan.sync()
    w = x.double().reshape(rows, cols)
    soft = torch.softmax(w, 1)
    want = soft + 0.75 * w
    # softmax: an argument of at most 12 log2 e rounded twice, exp2, at most 64 + 10 additions a term
    # takes part in, the quotient; then the product and the sum, a rounding each
    eps = 2.0 ** -24
    bound = eps * (soft * (74 + 2 * 18 + 6) + (0.75 * w).abs() + want.abs())
    err = (out.double().reshape(rows, cols) - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
