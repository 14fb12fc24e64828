"""kernels/matmul_dma.hip with operands of any extent and alignment: every tile it takes, ragged and whole
rows, columns and depths (the end of the depth 1, 33, 63 and 64 deep), odd and even strides along either axis, every
layout, operands that begin between two dwords.  Against the product in float64, element by element, within the
rounding of K fp32 additions (K * 2^-24 * sum of |a b|; the products of 16-bit values are exact)."""
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

SHAPES = [(513, 511, 1001, "bfloat16", "nn", "64x64"), (513, 497, 769, "bfloat16", "tn", "64x64"), (129, 1027, 769, "bfloat16", "nt", "64x64"), (703, 698, 704, "bfloat16", "nn", "64x64"),
          (702, 698, 894, "float16", "nt", "64x64"), (17, 9001, 799, "bfloat16", "tt", "64x64"), (1090, 1030, 161, "bfloat16", "nn", "64x128"),
          (1091, 1031, 127, "float16", "tn", "64x128"), (1500, 1400, 129, "bfloat16", "nt", "128x128"), (1503, 1401, 130, "bfloat16", "tt", "128x128"),
          (2050, 2100, 130, "bfloat16", "tn", "128x256"), (2049, 2101, 191, "bfloat16", "nt", "128x256"), (3000, 3001, 33, "bfloat16", "nn", "64x128"),
          (3001, 2999, 32, "bfloat16", "tn", "64x128")]


def _case(m, n, k, dtype, layout, tile):
    return dict(kind="matmul", m=m, n=n, k=k, dtype=dtype, layout=layout)


def _is_it(desc, tile):
    return f"tile {tile}x64 " in desc and "rows of any alignment" in desc


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_stays_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    it = s.items[0]
    assert _is_it(_ffi.take_string(hiplib.poly_hip_describe(it.root, PLAN)), c[5])
    assert "rows of any alignment" not in _ffi.take_string(hiplib.poly_hip_describe(it.root, 0))
    check_as_of_a_plan(hiplib, s, it)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", [SHAPES[0][:5], SHAPES[9][:5], (1030, 1040, 97, "float32", "nn"), (1801, 1700, 160, "float32", "tn")], ids=lambda c: "-".join(map(str, c)))
def test_candidates_for_tuning_stay_in_bounds(c, hiplib, monkeypatch):
    """The other tiles that the on-device search times."""
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    monkeypatch.setenv("POLY_BEAM", "1")
    pf = cases._matmul_schedule(_case(*c, None)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    it = s.items[0]
    variants = _ffi.take_string(hiplib.poly_hip_render(it.root, b"k", PLAN, None)).split("\n// ---- variant ")[1:]
    assert len(variants) >= (1 if c[3] == "float32" else 3)
    sizes = [s.buf_slots[it.buf_slot_indices[p]].nbytes for p in range(it.n_buf_slots)]
    for v in variants:
        label, source = v.split("\n", 1)
        bm, bn, wm, wn = map(int, re.match(r"(?:f32_)?(\d+)x(\d+)\w*?w(\d)x(\d)", label).groups())
        grid = (-(-c[0] // bm) * -(-c[1] // bn), 1, 1)
        hostcheck.check_kernel(source, hostcheck._entry_name(source), grid, 64 * wm * wn, sizes, block_stride=max(1, grid[0] * 64 * wm * wn // (1 << 16)))


@pytest.mark.gpu
@pytest.mark.parametrize("between_dwords", [False, True])
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_against_float64(c, between_dwords):
    import torch
    m, n, k, dtype, layout, tile = c
    state = cases.prepare(_case(*c), 5)
    assert _is_it(state["plan"].kernel_info()[0]["desc"], tile)
    ab = {}
    for s in state["plan"].external_slots():
        if s.name in "AB":
            t = state["data"][s.index]
            if between_dwords:
                t = torch.cat([t.new_full((1,), float("nan")), t, t.new_full((1,), float("nan"))])[1:-1]
                state["data"][s.index] = t
            ab[s.name] = t.double().cpu()
    got = cases.run(state)["C"]
    state["plan"].sync()
    a = ab["A"].reshape(k, m).T if layout[0] == "t" else ab["A"].reshape(m, k)
    b = ab["B"].reshape(n, k).T if layout[1] == "t" else ab["B"].reshape(k, n)
    err = (got.double().cpu().reshape(m, n) - a @ b).abs()
    bound = k * 2.0 ** -24 * (a.abs() @ b.abs())
    assert bool((err <= bound).all()), float((err / bound).max())
