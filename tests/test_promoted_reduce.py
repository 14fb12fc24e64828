"""Reductions of reductions to few outputs in two stages, the second a wave per output: the fewest and
most outputs, the fewest terms, one more, and many; every output on a wave of its own.  Against float64 on the host."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SIZES = [(1, 64, 256), (1, 65, 300), (3, 127, 257), (5, 4096, 256), (64, 70, 256), (33, 1000, 256)]


def _plan(op, rows, terms, inner):
    """out[r] = op over t of w[t] * (sum over k of x[r, t, k])"""
    s = cases.Schedule()
    out, x, w = s.buf("out", rows), s.buf("x", rows * terms * inner), s.buf("w", terms)
    (r,) = s.ranges(rows)
    t = s.rrange(terms)
    k = s.rrange(inner)
    s.store(out, r, s.reduce(op, w[t] * s.reduce("ADD", x[(r * terms + t) * inner + k], k), t), r) if rows > 1 else \
        s.store(out, 0, s.reduce(op, w[t] * s.reduce("ADD", x[t * inner + k], k), t))
    return s.plan()


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("op", ["ADD", "MAX"])
@pytest.mark.parametrize("rows,terms,inner", SIZES)
def test_in_bounds(op, rows, terms, inner, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _plan(op, rows, terms, inner)
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert "two stages" in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    launch = (C.c_int * 8)()
    _ffi.take_string(hiplib.poly_hip_render(s.items[0].root, b"k", 0, launch))
    assert launch[0] == (rows + 3) // 4 and launch[3] == 256      # of the second stage: four waves to a workgroup
    assert hostcheck.check_schedule(hiplib, pf.schedule) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ADD", "MAX"])
@pytest.mark.parametrize("rows,terms,inner", SIZES)
def test_against_float64(op, rows, terms, inner):
    import torch
    plan = _plan(op, rows, terms, inner)
    g = torch.Generator(device="cuda").manual_seed(rows * terms)
    by = {"x": torch.randn(rows * terms * inner, device="cuda", generator=g), "w": torch.rand(terms, device="cuda", generator=g) + 0.5,
          "out": torch.empty(rows, device="cuda")}
    data = [None] * len(plan.slots)
    for s in plan.external_slots():
        data[s.index] = by[s.name]
    plan.run(data)
    plan.sync()
    x, w = by["x"].double().reshape(rows, terms, inner), by["w"].double()
    each, size = w * x.sum(2), w * x.abs().sum(2)
    # a rounding per addition: inner ones, and terms / 64 + 6 of the terms'; one per product
    eps = 2.0 ** -24
    want, bound = (each.sum(1), size.sum(1) * eps * (inner + terms / 64 + 8)) if op == "ADD" else (each.max(1).values, size.max(1).values * eps * (inner + 2))
    assert bool(((by["out"].double() - want).abs() <= bound).all())
