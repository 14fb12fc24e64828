"""A LayerNorm in front of a product that writes what the LayerNorm reads: such rows are not computed by
the product, whose workgroups would read them while others store.  Stored straight into the rows, added
to them, copied back into them, and rows that are an intermediate; beside them the forms with an output
of its own, which are one launch.  And the same bits as with a launch for the LayerNorm."""
import ctypes as C
import os
import sys

import pytest

from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

F32 = cases.F32
SIZES = [(12, 768, "bfloat16"), (24, 768, "bfloat16"), (8, 768, "float32")]
# what the product's result goes to, and whether the rows are computed by it ("copy plus": the sum has a
# buffer of its own, which is copied into the rows by a launch behind it)
FORMS = [("out", True), ("x", False), ("x plus", False), ("out plus", True), ("copy", False), ("copy plus", True), ("copy beside", True), ("intermediate", False)]


def _schedule(rows, d, w, form):
    s = cases.Schedule()
    x, weight, bias, gamma, beta = s.buf("x", rows * d, w), s.buf("weight", d * d, w), s.buf("bias", d, w), s.buf("gamma", d, w), s.buf("beta", d, w)
    out = s.buf("out", rows * d, w)
    src = x
    if form == "intermediate":
        (i,) = s.ranges(rows * d)
        src = s.store(s.tmp(rows * d, w), i, x[i] * 0.5, i)
    (q,) = s.ranges(rows)
    k = s.rrange(d)
    mean = s.store(s.tmp(rows), q, s.reduce("ADD", src[q * d + k].cast(F32), k) / float(d), q)
    (q,) = s.ranges(rows)
    k = s.rrange(d)
    e = src[q * d + k].cast(F32) + (-mean[q])
    var = s.store(s.tmp(rows), q, s.reduce("ADD", e * e, k) / float(d), q)
    q, j = s.ranges(rows, d)
    y = ((src[q * d + j].cast(F32) + (-mean[q])) * (var[q] + 1e-5).un("SQRT").un("RECIPROCAL")).cast(w)
    y = s.store(s.tmp(rows * d, w), q * d + j, y * gamma[j] + beta[j], q, j)

    def linear(dst):
        q, j = s.ranges(rows, d)
        k = s.rrange(d)
        acc = s.reduce("ADD", y[q * d + k].cast(F32) * weight[k * d + j].cast(F32), k).cast(w)
        return s.store(dst, q * d + j, acc + bias[j], q, j)

    def elementwise(dst, value):
        (i,) = s.ranges(rows * d)
        return s.store(dst, i, value(i), i)

    if form in ("out", "x"):
        linear(out if form == "out" else x)
    elif form == "intermediate":
        linear(src)
        elementwise(out, lambda i: src[i] * 2.0)
    else:
        v = linear(s.tmp(rows * d, w))
        if form.endswith("plus"):
            v = elementwise(dict(x=x, out=out).get(form.split()[0]) or s.tmp(rows * d, w), lambda i, v=v: x[i] + v[i])
        if form.startswith("copy"):
            elementwise(out if form == "copy beside" else x, lambda i: v[i])
    return s


@pytest.mark.parametrize("form,fused", FORMS)
@pytest.mark.parametrize("rows,d,w", SIZES)
def test_grouping(rows, d, w, form, fused, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _schedule(rows, d, w, form).plan()
    found = 0
    for gi in range(hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None)):
        src = C.c_void_p()
        hiplib.poly_hip_fused_groups(pf.schedule, gi, C.byref(src), None)
        text = _ffi.take_string(src.value)
        if "#define POLY_A_ROWS(" not in text:
            continue
        found += 1
        # (positions in the rows' own array, never a pointer in front of it)
        assert text.count("const PolyRowsOut data0") == 1
        assert hiplib.poly_hip_compile_check(text.split("\n// ---- ")[0].encode()) == 0
        slots = (C.c_int * 64)()
        n = hiplib.poly_hip_fused_group_launch(pf.schedule, gi, slots, 64, None)
        assert slots[0] not in list(slots[1:n]), list(slots[:n])
    assert found == int(fused)


def _run(rows, d, w, form):
    import torch
    plan = _schedule(rows, d, w, form).plan()
    g = torch.Generator(device="cuda").manual_seed(rows)
    by, data = {}, [None] * len(plan.slots)
    for slot in plan.external_slots():
        scale = dict(weight=d ** -0.5, bias=0.02, beta=0.02).get(slot.name, 1.0)
        by[slot.name] = data[slot.index] = (torch.randn(slot.numel, generator=g, device="cuda") * scale).to(getattr(torch, w))
    seen = []
    for _ in range(3):
        plan.run(data)
        seen.append({k: v.cpu().view(torch.uint8).numpy().tobytes() for k, v in by.items()})
    return seen, sum("compute A's rows" in k["desc"] for k in plan.kernel_info())


@pytest.mark.gpu
@pytest.mark.parametrize("form,fused", FORMS)
@pytest.mark.parametrize("rows,d,w", SIZES)
def test_same_bits(rows, d, w, form, fused, monkeypatch):
    here, n = _run(rows, d, w, form)
    monkeypatch.setenv("POLY_HIP_NO_ROWS_IN_PRODUCT", "1")
    there, n_there = _run(rows, d, w, form)
    assert (n, n_there) == (int(fused), 0)
    assert here == there


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["out", "out plus", "copy beside"])
@pytest.mark.parametrize("rows,d,w", SIZES)
def test_output_bound_over_the_rows(rows, d, w, form, monkeypatch):
    """The caller's own output over the rows that the LayerNorm reads, as a whole and from the middle on (not
    where the rows are added to the result: that reads them where the output is written): the bits of
    a plan that launches the LayerNorm by itself, before and after passes on buffers apart."""
    import torch

    def run():
        plan = _schedule(rows, d, w, form).plan()
        g = torch.Generator(device="cuda").manual_seed(rows)
        by, data = {}, [None] * len(plan.slots)
        for slot in plan.external_slots():
            scale = dict(weight=d ** -0.5, bias=0.02, beta=0.02).get(slot.name, 1.0)
            n = slot.numel + (slot.numel // 2 if slot.name == "x" else 0)
            by[slot.name] = (torch.randn(n, generator=g, device="cuda") * scale).to(getattr(torch, w))
            data[slot.index] = by[slot.name][:slot.numel]
        out, n = [s.index for s in plan.external_slots() if s.name == "out"][0], rows * d
        seen = []
        middle = [] if form == "out plus" else [by["x"][n // 2:]]
        for bound in [data[out], by["x"][:n], data[out]] + middle + [by["x"][:n], data[out]]:
            data[out] = bound
            plan.run(data)
            seen += [v.cpu().view(torch.uint8).numpy().tobytes() for v in (by["x"], bound)]
        return seen, sum("compute A's rows" in k["desc"] for k in plan.kernel_info())

    here, n = run()
    monkeypatch.setenv("POLY_HIP_NO_ROWS_IN_PRODUCT", "1")
    monkeypatch.setenv("POLY_HIP_NO_COPY_DROP", "1")
    there, n_there = run()
    assert (n, n_there) == (1, 0)
    assert here == there
