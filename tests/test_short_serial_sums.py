"""Sums that one thread adds up term by term, about the extents where all loads of a loop, those of as many
terms as divide it, of sixteen or of eight are in flight: column sums and sums of products, few and many outputs.  Against float64 on the host."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_promoted_reduce import cases

# columns, terms, whether two operands are read a term, how the loop is unrolled
SIZES = [(100, 15, False, ""), (100, 16, False, "unroll"), (1290, 33, True, "unroll 11"), (70, 36, True, "unroll 12"), (70, 37, True, "unroll 16"), (70, 28, True, "unroll"),
         (70, 29, True, "unroll 16"), (100000, 32, True, "unroll 16"), (257, 56, False, "unroll"), (257, 57, False, "unroll 16"), (257, 63, False, "unroll 9"), (257, 64, False, "unroll 8"),
         (70001, 17, True, "unroll")]


def _plan(cols, terms, two):
    """out[i] = sum over r of x[r, i] (+ y[r, i])"""
    s = cases.Schedule()
    out, x, y = s.buf("out", cols), s.buf("x", terms * cols), s.buf("y", terms * cols)
    (i,) = s.ranges(cols)
    r = s.rrange(terms)
    s.store(out, i, s.reduce("ADD", x[r * cols + i] + y[r * cols + i] if two else x[r * cols + i], r), i)
    return s.plan()


@pytest.mark.parametrize("cols,terms,two,how", SIZES)
def test_route(cols, terms, two, how, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _plan(cols, terms, two)
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    launch = (C.c_int * 8)()
    source = _ffi.take_string(hiplib.poly_hip_render(s.items[0].root, b"k", 0, launch))
    body = source[source.rfind("__global__"):]
    pragmas = [line.strip() for line in body.splitlines() if "#pragma" in line]
    assert pragmas == (["#pragma " + how] if how else []), body
    if os.path.exists(hostcheck.CLANG):
        assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("cols,terms,two,how", SIZES)
def test_against_float64(cols, terms, two, how):
    import torch
    plan = _plan(cols, terms, two)
    g = torch.Generator(device="cuda").manual_seed(cols + terms)
    by = {n: torch.randn(terms * cols, device="cuda", generator=g) for n in "xy"}
    by["out"] = torch.empty(cols, device="cuda")
    data = [None] * len(plan.slots)
    for s in plan.external_slots():
        data[s.index] = by[s.name]
    plan.run(data)
    plan.sync()
    x, y = (by[n].double().reshape(terms, cols) for n in "xy")
    each, size = (x + y, x.abs() + y.abs()) if two else (x, x.abs())
    # a rounding per addition
    assert bool(((by["out"].double() - each.sum(0)).abs() <= size.sum(0) * 2.0 ** -24 * (terms + 1)).all())
