"""LayerNorms over up to 64 rows computed by the product behind them: whole models of one row, of
odd numbers of rows, of whole tiles of 16 and of one row more, in bf16 (two rows to a wave) and fp32,
give the bits they give with a launch for each LayerNorm; 65 rows, and fp32 tiles that would have four rows
to a wave, keep the launches."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SIZES = [(1, 2, "bfloat16", 768, 4), (1, 12, "bfloat16", 768, 4), (3, 5, "bfloat16", 768, 4), (2, 8, "float32", 768, 4), (1, 7, "float32", 768, 4), (1, 16, "bfloat16", 768, 4),
         (1, 11, "bfloat16", 256, 4), (1, 17, "bfloat16", 768, 4), (3, 21, "bfloat16", 768, 4),
         (1, 64, "bfloat16", 768, 4), (1, 65, "bfloat16", 768, 0), (1, 17, "float32", 768, 0), (1, 5, "float32", 1024, 0)]


def _case(batch, ctx, dtype, d_model):
    return cases._gpt2(batch, ctx, dtype, layers=2, heads=d_model // 64, d_model=d_model)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("batch,ctx,dtype,d_model,fused", SIZES)
def test_in_bounds(batch, ctx, dtype, d_model, fused, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._gpt2_schedule(_case(batch, ctx, dtype, d_model)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    found = 0
    for gi in range(hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None)):
        src = C.c_void_p()
        hiplib.poly_hip_fused_groups(pf.schedule, gi, C.byref(src), None)
        text = _ffi.take_string(src.value)
        if "#define POLY_A_ROWS(" not in text:
            continue
        found += 1
        slots, launch = (C.c_int * 64)(), (C.c_int * 4)()
        n = hiplib.poly_hip_fused_group_launch(pf.schedule, gi, slots, 64, launch)
        sizes = [int(s.buf_slots[slots[i]].nbytes) for i in range(n)]
        if found <= 2:
            hostcheck.check_kernel(text.split("\n// ---- ")[0], "poly_k", tuple(launch[:3]), launch[3], sizes)
    assert found == fused


@pytest.mark.gpu
@pytest.mark.parametrize("batch,ctx,dtype,d_model,fused", SIZES)
def test_same_bits(batch, ctx, dtype, d_model, fused, monkeypatch):
    import torch

    def logits():
        state = cases.prepare(_case(batch, ctx, dtype, d_model), 3)
        n = sum("compute A's rows" in k["desc"] for k in state["plan"].kernel_info())
        outs = []
        for _ in range(3):
            cases.run(state)
            state["plan"].sync()
            outs.append(state["out"]["output"].clone())
        assert all(torch.equal(outs[0], o) for o in outs) and bool(torch.isfinite(outs[0].float()).all())
        return outs[0], n

    here, n = logits()
    monkeypatch.setenv("POLY_HIP_NO_ROWS_IN_PRODUCT", "1")
    there, n_there = logits()
    assert (n, n_there) == (fused, 0)
    assert torch.equal(here, there)
