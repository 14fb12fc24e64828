"""Products whose operands are views, on every template a plan's products run on, both operands and both ways they can
lie: rows or the depth in reverse order, which an operand's offsets run down; slices of wider buffers, whose rows begin
between two dwords or 16 bytes and end inside a tile, behind whole 8 elements or not; rows far apart, in buffers
of 4 GiB and more; batches of matrices.  On the host with buffers of their exact size, and against the product in float64, element by
element, within the rounding of K fp32 additions and products (K * 2^-24 * sum of |a b|)."""
import ctypes as C
import os
import re
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_f32_planes import PLAN, check_as_of_a_plan

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

F32_PLANES, RING, DMA, REGISTERS, WAVES = "three planes of each f32 value", "rows of any alignment", "straight into LDS", "32x32x16", "depth dealt to"
REVERSED = [(1793, 1664, 129, "float32", "nn", "A rows", F32_PLANES), (1665, 1793, 191, "float32", "nt", "B rows", F32_PLANES), (1665, 1793, 191, "float32", "nt", "A rows B rows", F32_PLANES),
            (1025, 1024, 65, "float32", "nt", "A rows B rows", F32_PLANES), (1024, 1024, 2048, "float32", "nt", "A rows B rows", F32_PLANES),
            (513, 511, 1001, "bfloat16", "nn", "A rows", RING), (1091, 1030, 161, "float16", "nt", "A rows B rows", RING), (1502, 1400, 130, "bfloat16", "nt", "A rows B rows", RING),
            (1152, 1024, 1536, "bfloat16", "nn", "A rows", DMA), (1152, 1024, 1536, "bfloat16", "tn", "A depth", DMA), (1152, 1024, 1536, "bfloat16", "nn", "B depth", DMA),
            (4096, 4096, 512, "float16", "nt", "A rows B rows", DMA), (2304, 512, 1536, "bfloat16", "nt", "B rows", DMA), (512, 512, 16384, "bfloat16", "nt", "A rows B rows", DMA),
            (49452, 1000, 512, "bfloat16", "nt", "A rows B rows", DMA), (16384, 64, 512, "bfloat16", "nt", "A rows B rows", REGISTERS),
            (40, 768, 512, "bfloat16", "nt", "A rows B rows", WAVES), (40, 768, 512, "float32", "nt", "A rows B rows", WAVES)]
# ("A 1003 1": rows of A, or where it lies along its rows depths of it, are 1003 elements apart, the first at 1)
SLICED = [(513, 520, 1001, "bfloat16", "nn", "B 521 0", RING), (513, 520, 1001, "bfloat16", "nn", "B 522 1", RING), (520, 513, 1001, "float16", "tn", "A 521 1", RING),
          (520, 504, 769, "bfloat16", "tt", "A 521 3 B 771 1", RING), (1096, 1032, 161, "bfloat16", "tn", "A 1099 0 B 1033 0", RING), (1111, 1000, 1501, "bfloat16", "nn", "B 1001 1", RING),
          (1400, 1504, 129, "bfloat16", "tn", "A 1401 5 B 1506 1", RING), (2056, 2104, 130, "float16", "tn", "A 2057 0 B 2106 1", RING), (3000, 3008, 33, "bfloat16", "nn", "A 35 1 B 3009 0", RING),
          (512, 514, 1001, "bfloat16", "nn", "B 515 1", RING), (1030, 1040, 97, "float32", "nn", "A 99 1 B 1056 3", F32_PLANES), (1801, 1700, 160, "float32", "tn", "A 1805 2 B 1701 1", F32_PLANES),
          (1152, 1024, 1536, "bfloat16", "nt", "A 1538 2 B 1544 8", DMA), (1152, 1024, 1536, "bfloat16", "tn", "A 1156 4 B 1026 2", DMA),
          (1152, 1024, 1536, "bfloat16", "nn", "A 1537 1 B 1025 0", DMA), (1152, 1024, 1536, "float16", "tn", "A 1153 0 B 1024 1", DMA), (4096, 4096, 512, "bfloat16", "nt", "A 513 1 B 515 2", DMA),
          (2304, 512, 1536, "bfloat16", "nt", "A 1537 0 B 1539 3", DMA), (512, 512, 16384, "bfloat16", "nn", "B 513 1", DMA), (16384, 64, 512, "bfloat16", "nn", "A 513 1 B 65 1", REGISTERS)]
# (of 2^30 elements and more, in 1.1 million from one row to the next)
FAR = [(1793, 1664, 129, "float32", "nn", "A 1100000 1", F32_PLANES), (1665, 1921, 191, "float32", "nt", "B 1100003 2", F32_PLANES), (1025, 1024, 65, "float32", "nn", "A 1100000 0", F32_PLANES),
       (1001, 1696, 1930, "float32", "tn", "A 1100000 0", F32_PLANES), (1090, 1941, 161, "bfloat16", "nt", "B 1100001 1", RING), (1152, 1024, 1920, "bfloat16", "nn", "B 1100000 0", DMA)]


def _is_it(desc, template):
    return template in desc and (template != REGISTERS or not any(t in desc for t in (F32_PLANES, RING, DMA)))


def _slice(name, view, rows, k, along_k):
    """Outer extent, inner extent, elements from one outer index to the next and the first element."""
    outer, inner = (rows, k) if along_k else (k, rows)
    given = re.search(name + r" (\d+) (\d+)", view)
    pitch, first = (int(given.group(1)), int(given.group(2))) if given else (inner, 0)
    return outer, inner, pitch, first


def schedule(m, n, k, dtype, layout, view):
    """C = A B, A and B buffers that end with their last element, read as `view` says."""
    s = cases.Schedule()

    def buf(name, rows, along_k):
        outer, inner, pitch, first = _slice(name, view, rows, k, along_k)
        return s.buf(name, first + (outer - 1) * pitch + inner, dtype)

    out, a, b = s.buf("C", m * n), buf("A", m, layout[0] == "n"), buf("B", n, layout[1] == "t")
    (r,) = s.ranges(m * n)
    x = s.rrange(k)

    def at(name, row, rows, along_k):
        row = row * -1 + (rows - 1) if name + " rows" in view else row
        d = x * -1 + (k - 1) if name + " depth" in view else x
        _, _, pitch, first = _slice(name, view, rows, k, along_k)
        return (row * pitch + d if along_k else d * pitch + row) + first

    s.store(out, r, s.reduce("ADD", a[at("A", r // n, m, layout[0] == "n")].cast(cases.F32) * b[at("B", r % n, n, layout[1] == "t")].cast(cases.F32), x), r)
    return s


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", REVERSED + SLICED, ids=lambda c: "-".join(map(str, c)))
def test_stays_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = schedule(*c[:6]).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert _is_it(_ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, PLAN)), c[6])
    check_as_of_a_plan(hiplib, s, s.items[0])


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", FAR, ids=lambda c: "-".join(map(str, c)))
def test_far_rows_are_those_read(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    m, n, k, dtype, layout, view, template = c
    pf = schedule(*c[:6]).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert _is_it(_ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, PLAN)), template)
    name = view[0]
    outer, inner, pitch, first = _slice(name, view, *((m, k, layout[0] == "n") if name == "A" else (n, k, layout[1] == "t")))
    size = 4 if dtype == "float32" else 2
    check_as_of_a_plan(hiplib, s, s.items[0], pieces={1 if name == "A" else 2: (first * size, inner * size, pitch * size, outer)})


@pytest.mark.gpu
@pytest.mark.parametrize("c", REVERSED + SLICED + FAR, ids=lambda c: "-".join(map(str, c)))
def test_against_float64(c):
    import torch
    from polygrad_amd.inputs import torch_dtype
    m, n, k, dtype, layout, view, template = c
    plan, g = schedule(*c[:6]).plan(), torch.Generator(device="cuda")
    g.manual_seed(6)
    assert _is_it(plan.kernel_info()[0]["desc"], template)
    data, by = [None] * len(plan.slots), {}
    for slot in plan.external_slots():
        t = torch.zeros(slot.numel, dtype=torch_dtype(slot.dtype), device="cuda")
        data[slot.index] = by[slot.name] = t if slot.numel > 1 << 28 else t.copy_(torch.randn(slot.numel, generator=g, device="cuda"))

    def operand(name, rows, along_k):
        outer, inner, pitch, first = _slice(name, view, rows, k, along_k)
        t = torch.as_strided(by[name], (outer, inner), (pitch, 1), first)
        if by[name].numel() > 1 << 28:      # (a few elements of it are all that is random)
            t.copy_(torch.randn((outer, inner), generator=g, device="cuda"))
        t = t.double()
        t = t if along_k else t.T
        return t.flip([d for d, axis in enumerate(("rows", "depth")) if f"{name} {axis}" in view])

    a, b = operand("A", m, layout[0] == "n"), operand("B", n, layout[1] == "t").T
    torch.cuda.synchronize()
    plan.run(data)
    plan.sync()
    err = (by["C"].double().reshape(m, n) - a @ b).abs()
    assert bool((err <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all())


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(1030, 1041, 97, "float32", "nn", "A 99 1 B 1056 3", F32_PLANES), (1801, 1703, 160, "float32", "tn", "A 1805 2 B 1709 1", F32_PLANES)],
                         ids=lambda c: "-".join(map(str, c)))
def test_what_lies_between_rows_changes_no_bit(c):
    """Not the values that three planes do not hold either, which send a tile another way."""
    import torch
    m, n, k, dtype, layout, view, template = c
    plan, g, outputs = schedule(*c[:6]).plan(), torch.Generator(device="cuda"), []
    assert _is_it(plan.kernel_info()[0]["desc"], template)
    for between in (0.0, 1e-40, float("nan"), float("inf")):
        g.manual_seed(7)
        data = [None] * len(plan.slots)
        for slot in plan.external_slots():
            data[slot.index] = t = torch.full((slot.numel,), between, device="cuda")
            if slot.name != "C":
                outer, inner, pitch, first = _slice(slot.name, view, m if slot.name == "A" else n, k, layout[0] == "n" if slot.name == "A" else layout[1] == "t")
                torch.as_strided(t, (outer, inner), (pitch, 1), first).copy_(torch.randn((outer, inner), generator=g, device="cuda"))
            else:
                outputs.append(t)
        torch.cuda.synchronize()
        plan.run(data)
        plan.sync()
    assert all(torch.equal(outputs[0], o) for o in outputs[1:])


# (batch, rows, columns, depth, dtype, layout, elements from one matrix of A to the next and of B, template; 0: the same for
# the whole batch, below 0: the batch in reverse order)
BATCHED = [(3, 400, 501, 601, "bfloat16", "nn", 400 * 601 + 1, 601 * 501 + 3, RING), (3, 400, 504, 601, "bfloat16", "nn", -400 * 601, 601 * 504 + 1, RING), (2, 520, 520, 769, "float16", "tt", 520 * 769 + 1, -520 * 769, RING),
           (3, 401, 1031, 161, "bfloat16", "nn", 401 * 161 + 7, 0, RING), (3, 385, 1031, 161, "bfloat16", "nt", -385 * 161 - 1, 0, RING), (3, 384, 512, 1024, "bfloat16", "nn", -384 * 1024, 1024 * 512 + 2, DMA),
           (4, 512, 512, 1024, "bfloat16", "nt", -512 * 1024, 0, DMA), (3, 600, 1664, 160, "float32", "nn", 600 * 160 + 3, 0, F32_PLANES), (3, 600, 1664, 161, "float32", "nt", -600 * 161, 0, F32_PLANES)]


def _batched_schedule(z, m, n, k, dtype, layout, za, zb, template):
    s = cases.Schedule()
    out, a, b = s.buf("C", z * m * n), s.buf("A", (z - 1) * abs(za) + m * k, dtype), s.buf("B", (z - 1) * abs(zb) + k * n, dtype)
    q, r = s.ranges(z, m * n)
    x = s.rrange(k)

    def at(row, rows, along_k, step):
        first = q * step + (1 - z) * step if step < 0 else q * step
        return first + (row * k + x if along_k else x * rows + row)

    s.store(out, q * (m * n) + r, s.reduce("ADD", a[at(r // n, m, layout[0] == "n", za)].cast(cases.F32) * b[at(r % n, n, layout[1] == "t", zb)].cast(cases.F32), x), q, r)
    return s


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", BATCHED, ids=lambda c: "-".join(map(str, c)))
def test_batched_stays_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _batched_schedule(*c).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert _is_it(_ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, PLAN)), c[8])
    check_as_of_a_plan(hiplib, s, s.items[0])


@pytest.mark.gpu
@pytest.mark.parametrize("c", BATCHED, ids=lambda c: "-".join(map(str, c)))
def test_batched_against_float64(c):
    import torch
    from polygrad_amd.inputs import torch_dtype
    z, m, n, k, dtype, layout, za, zb, template = c
    plan, g = _batched_schedule(*c).plan(), torch.Generator(device="cuda")
    g.manual_seed(8)
    assert _is_it(plan.kernel_info()[0]["desc"], template)
    data, by = [None] * len(plan.slots), {}
    for slot in plan.external_slots():
        data[slot.index] = by[slot.name] = torch.randn(slot.numel, generator=g, device="cuda").to(torch_dtype(slot.dtype))
    torch.cuda.synchronize()
    plan.run(data)
    plan.sync()
    for i in range(z):
        def matrix(name, rows, cols, step):
            return torch.as_strided(by[name], (rows, cols), (cols, 1), (z - 1 - i if step < 0 else i) * abs(step)).double()
        a = matrix("A", m, k, za) if layout[0] == "n" else matrix("A", k, m, za).T
        b = matrix("B", k, n, zb) if layout[1] == "n" else matrix("B", n, k, zb).T
        err = (by["C"].double().reshape(z, m, n)[i] - a @ b).abs()
        assert bool((err <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all())
