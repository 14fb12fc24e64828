"""Switches that take a mechanism away take it away from every template that has it:
POLY_HIP_NO_F32_MFMA from fp32 products and fp32 attention, POLY_HIP_NO_SPLIT_K from fp32
products whose depth goes to several workgroups, POLY_HIP_NO_ATTENTION_ROWS the attention of
any length, POLY_HIP_NO_ROW_CHAIN_SIZES the row chains of short and of long rows."""
import ctypes as C

import pytest

from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, cases


def _described(case, hiplib, monkeypatch):
    """(every item of the case's schedule, every group of the plan), as text."""
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._SCHEDULES[case["kind"]](case).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    items = [_ffi.take_string(hiplib.poly_hip_describe(s.items[i].root, 0)) for i in range(s.n_items)]
    groups = []
    for g in range(hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None)):
        src = C.c_void_p()
        hiplib.poly_hip_fused_groups(pf.schedule, g, C.byref(src), None)
        groups.append(_ffi.take_string(src.value))
    return items, groups


@pytest.mark.parametrize("shape", [(12, 768, 3072), (300, 64, 4096), (1024, 1024, 1024)])
def test_no_f32_mfma_in_products(shape, hiplib, monkeypatch):
    case = _case(*shape, "float32", "nn")
    assert "16x16x4 f32" in _described(case, hiplib, monkeypatch)[0][0]
    monkeypatch.setenv("POLY_HIP_NO_F32_MFMA", "1")
    assert "mfma" not in _described(case, hiplib, monkeypatch)[0][0]


def test_no_f32_mfma_in_attention(hiplib, monkeypatch):
    case = cases._gpt2(1, 40, "float32", layers=1)
    assert any("POLY_FA_M" in g for g in _described(case, hiplib, monkeypatch)[1])
    monkeypatch.setenv("POLY_HIP_NO_F32_MFMA", "1")
    items, groups = _described(case, hiplib, monkeypatch)
    assert not any("POLY_FA_M" in g or "POLY_MFMA_F32" in g for g in groups) and not any("mfma" in i for i in items)


@pytest.mark.parametrize("shape", [(32, 512, 4096), (300, 10, 8192)])
def test_no_split_k(shape, hiplib, monkeypatch):
    case = _case(*shape, "float32", "nn")
    assert "K dealt to" in _described(case, hiplib, monkeypatch)[0][0]
    monkeypatch.setenv("POLY_HIP_NO_SPLIT_K", "1")
    assert "K dealt to" not in _described(case, hiplib, monkeypatch)[0][0]


def test_no_attention_rows(hiplib, monkeypatch):
    case = cases._gpt2(1, 40, "bfloat16", layers=1)
    assert any("attention_rows.hip" in g for g in _described(case, hiplib, monkeypatch)[1])
    monkeypatch.setenv("POLY_HIP_NO_ATTENTION_ROWS", "1")
    assert not any("attention_rows.hip" in g for g in _described(case, hiplib, monkeypatch)[1])


def _largest_group(cols, hiplib):
    """Kernels of the largest fused group of a softmax over rows of `cols` computed elements."""
    pf = cases._rows_schedule(dict(kind="rows", op="softmax", rows=3, cols=cols)).plan()
    most, n = 0, C.c_int()
    for g in range(hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None)):
        src = C.c_void_p()
        hiplib.poly_hip_fused_groups(pf.schedule, g, C.byref(src), C.byref(n))
        _ffi.take_string(src.value)
        most = max(most, n.value)
    return most


@pytest.mark.parametrize("cols", [31, 1025, 50257])
def test_no_row_chain_sizes(cols, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    assert _largest_group(cols, hiplib) == 4
    monkeypatch.setenv("POLY_HIP_NO_ROW_CHAIN_SIZES", "1")
    assert _largest_group(cols, hiplib) < 4
