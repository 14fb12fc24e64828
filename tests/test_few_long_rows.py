"""Sums and maxima over a few long rows, sixteen waves to a row: one vector a lane and many, ragged ends, rows that begin on
no vector, the most and one more than the most rows that are dealt out so.  Sums against float64 within the rounding of
the additions on the way of a term (its lane's, six across the lanes of a wave, four across the waves) and the chain's."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SHAPES = [(1, 4096, True), (2, 4097, True), (3, 16387, True), (7, 50257, True), (400, 4100, True), (401, 4100, False), (5, 4095, False)]


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("op", ["sum", "max"])
@pytest.mark.parametrize("rows,cols,wide", SHAPES)
def test_stays_in_bounds(rows, cols, wide, op, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._rows_schedule(dict(kind="rows", op=op, rows=rows, cols=cols)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert ("G=1024" in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))) == wide
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.parametrize("rows,operands,sines,wide", [(256, 4, 0, True), (257, 3, 0, True), (257, 4, 0, False), (400, 3, 0, True), (400, 6, 0, False), (64, 16, 0, True), (64, 17, 0, False), (64, 3, 3, True),
                                                      (64, 4, 4, False)])
def test_rows_of_many_operands(rows, operands, sines, wide, hiplib, monkeypatch):
    """More rows than CUs go to sixteen waves each only where a few operands are read, and none where a lane's registers
    would not hold what it reads."""
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    s = cases.Schedule()
    out, bufs = s.buf("out", rows), [s.buf(f"b{i}", rows * 4096) for i in range(operands)]
    (r,) = s.ranges(rows)
    k = s.rrange(4096)
    monkeypatch.setitem(cases._OPS, "SIN", 27)
    values = [b[r * 4096 + k].un("SIN") if i < sines else b[r * 4096 + k] for i, b in enumerate(bufs)]
    value = values[0]
    for v in values[1:]:
        value = value * v
    s.store(out, r, s.reduce("ADD", value, k), r)
    pf = s.plan()
    item = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents.items[0]
    assert ("G=1024" in _ffi.take_string(hiplib.poly_hip_describe(item.root, 0))) == wide


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["sum", "max"])
@pytest.mark.parametrize("rows,cols,wide", SHAPES)
def test_against_float64(rows, cols, wide, op):
    state = cases.prepare(dict(kind="rows", op=op, rows=rows, cols=cols), 3)
    assert ("G=1024" in state["plan"].kernel_info()[0]["desc"]) == wide
    got = cases.run(state)["out"]
    state["plan"].sync()
    by = {s.name: state["data"][s.index].double().reshape(rows, cols) for s in state["plan"].external_slots() if s.name != "out"}
    y = (by["a"] * by["b"] + by["c"]).exp2().clamp(-4, 4)
    want = y.sum(1) if op == "sum" else y.max(1).values
    steps = (cols + 255) // 256 + 12 if op == "sum" else 0
    # (the elements: two roundings of at most 3 in front of exp2, whose own error is within 2 units)
    bound = (steps + 8) * 2.0 ** -24 * (y.abs().sum(1) if op == "sum" else y.abs().max(1).values)
    assert bool(((got.double() - want).abs() <= bound).all())
