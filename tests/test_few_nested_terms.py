"""Reductions of reductions to few outputs of fewer than 128 terms, a wave per output: the fewest terms and
elements, one less of each, as many terms as lanes and one more, the most terms and outputs, one output
more.  Against float64 on the host."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_promoted_reduce import _plan, cases

# rows, terms, elements of a term, whether a wave adds them up
SIZES = [(1, 16, 8, True), (1, 15, 9, False), (1, 18, 7, False), (1, 33, 10, True), (4, 64, 3, True), (3, 65, 2, True), (64, 127, 257, True), (65, 127, 2, False)]


@pytest.mark.parametrize("op", ["ADD", "MAX"])
@pytest.mark.parametrize("rows,terms,inner,wave", SIZES)
def test_route(op, rows, terms, inner, wave, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _plan(op, rows, terms, inner)
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    text = _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    if inner < 256:      # (longer terms are dealt to two stages)
        assert text.startswith("row-reduce") == wave, text
    if os.path.exists(hostcheck.CLANG):
        assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ADD", "MAX"])
@pytest.mark.parametrize("rows,terms,inner,wave", SIZES)
def test_against_float64(op, rows, terms, inner, wave):
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
    # a rounding per addition of a term's elements and one per product; of the terms, at most one each
    eps = 2.0 ** -24
    want, bound = (each.sum(1), size.sum(1) * eps * (inner + terms + 2)) if op == "ADD" else (each.max(1).values, size.max(1).values * eps * (inner + 2))
    assert bool(((by["out"].double() - want).abs() <= bound).all())
