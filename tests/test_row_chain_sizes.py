"""Row chains that keep their row in registers (softmax and LayerNorm over a computed row) at
the sizes where the dealing of a row changes: below and at half a wave, at a wave, odd rows,
the most elements a lane of 64, 256 and 1024 lanes keeps and one more, the longest row that is
kept and one more, and the even rows beside them.  Against float64 on the host."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SIZES = [(5, 8), (9, 31), (70, 32), (3, 33), (33, 127), (1, 128), (2049, 1001), (5, 1023), (2050, 1024), (2049, 1025), (2048, 2050), (3, 4095), (7, 8191), (3, 8193), (2, 8194),
         (2, 16388), (2, 50257), (2, 53248), (1, 50257), (1, 53248)]
TOO_LONG = [(2, 53249)]


def _case(op, rows, cols):
    return dict(kind="rows", op=op, rows=rows, cols=cols)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("op", ["softmax", "layernorm"])
@pytest.mark.parametrize("rows,cols", SIZES + TOO_LONG)
def test_one_launch_in_bounds(op, rows, cols, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._rows_schedule(_case(op, rows, cols)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None) == 1
    src, n_items = C.c_void_p(), C.c_int()
    hiplib.poly_hip_fused_groups(pf.schedule, 0, C.byref(src), C.byref(n_items))
    text = _ffi.take_string(src.value)
    assert n_items.value == (2 if (rows, cols) in TOO_LONG else s.n_items)
    # (positions worked out again in each phase: where elements have an address each, or rows are many)
    assert ("asm volatile" in text) == (cols in (50257, 53248) and (rows, cols) != (1, 53248))
    slots, launch = (C.c_int * 64)(), (C.c_int * 4)()
    n = hiplib.poly_hip_fused_group_launch(pf.schedule, 0, slots, 64, launch)
    sizes = [int(s.buf_slots[slots[i]].nbytes) for i in range(n)]
    hostcheck.check_kernel(text.split("\n// ---- ")[0], "poly_k", tuple(launch[:3]), launch[3], sizes, block_stride=max(1, launch[0] * launch[3] >> 16))


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["softmax", "layernorm"])
@pytest.mark.parametrize("rows,cols", SIZES + TOO_LONG)
def test_against_float64(op, rows, cols):
    import torch
    state = cases.prepare(_case(op, rows, cols), 7)
    info = state["plan"].kernel_info()
    assert (rows, cols) in TOO_LONG or ["row chain of 4" in k["desc"] for k in info] == [True]
    cases.run(state)
    state["plan"].sync()
    by = {s.name: state["data"][s.index].double().cpu().reshape(-1, cols) for s in state["plan"].external_slots()}
    y = torch.exp2(by["a"] * by["b"] + by["c"]).clamp(-4, 4)
    eps = 2.0 ** -24
    # a lane adds at most 64 elements, then ten partial sums are added on the way to the total
    if op == "softmax":
        want = torch.softmax(y, 1)
        # terms: exp2 of an argument of at most 5.5 that was rounded three times, itself within 2 eps
        bound = want * eps * (74 + 3 * 5.5 + 4)
    else:
        d = y - y.mean(1, keepdim=True)
        dev = torch.sqrt((d * d).mean(1, keepdim=True) + 1e-5)
        want = d / dev
        # the mean of values up to 4 shifts every element; the deviation and the quotient scale it
        bound = eps * (74 + 4) * 4 / dev + want.abs() * eps * (74 + 8)
    err = (by["out"] - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
