"""Embeddings as masked sums over a table: the gather, and the walk over the whole table where the
buffer it is compared with is not 0, 1, 2 ..., are branches of one launch; tables of up to 2048 rows are
checked there too.  At and above that edge, fewer and more workgroups than the walk has, odd widths,
with a buffer that is right and with its first, its last or all its entries wrong; selected
rows are exact either way (one term, or a sum of zeros and one term)."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SIZES = [(64, 5, 33, "float32"), (345, 400, 64, "bfloat16"), (2048, 37, 48, "bfloat16"), (2049, 37, 48, "float32"), (3000, 9000, 128, "bfloat16")]


def _schedule(V, n, D, w):
    s = cases.Schedule()
    out, ids, ar, table = s.buf("out", n * D, w), s.buf("ids", n), s.buf("ar", V), s.buf("table", V * D, w)
    r, j = s.ranges(n, D)
    v = s.rrange(V)
    hit = cases.where(ids[r].ne(ar[v]), cases.const(0.0, "float32"), cases.const(1.0, "float32"))
    pick = cases.where(hit, table[v * D + j].cast("float32"), cases.const(0.0, "float32"))
    s.store(out, r * D + j, s.reduce("ADD", pick, v).cast(w), r, j)
    return s


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", [c for c in SIZES if c[0] <= 2048], ids=str)
def test_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _schedule(*c).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert "check, gather and fallback in one launch" in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert hostcheck.check_schedule(hiplib, pf.schedule) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("wrong", ["none", "first", "last", "all"])
@pytest.mark.parametrize("c", SIZES, ids=str)
def test_selected_rows(c, wrong):
    import torch
    V, n, D, w = c
    g = torch.Generator().manual_seed(V)
    plan = _schedule(*c).plan()
    info = plan.kernel_info()[0]
    assert info["klass"] == "gather"
    assert ("check, gather and fallback" if V <= 2048 else "gather and fallback in one launch") in info["desc"]
    table = torch.randn(V, D, generator=g).to(getattr(torch, w))
    ar = torch.arange(V).float()
    if wrong == "all":
        ar = ar[torch.randperm(V, generator=g)]
    elif wrong != "none":
        ar[0 if wrong == "first" else -1] = V + 7.0
    ids = torch.randint(0, V, (n,), generator=g).float()
    ids[:4] = torch.tensor([0.0, V - 1.0, V + 7.0, 0.5])
    want = (ids[:, None] == ar[None, :]).double() @ table.double()
    data = [None] * len(plan.slots)
    by = dict(out=torch.full((n * D,), 3.0, dtype=table.dtype).cuda(), ids=ids.cuda(), ar=ar.cuda(), table=table.cuda().reshape(-1))
    for sl in plan.external_slots():
        data[sl.index] = by[sl.name]
    for _ in range(3):
        plan.run(data)
        plan.sync()
        assert bool((by["out"].cpu().double().reshape(n, D) == want).all())
