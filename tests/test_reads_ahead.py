"""kernels/matmul_wave.hip with workgroups in front that read B ahead of the tiles: they stay
inside B on every layout, type and ragged edge, also where an XCD has no tile, and the tiles
behind them are the ones they were."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

SHAPES = [(12, 33, 40, "bfloat16", "nn"), (17, 31, 255, "bfloat16", "nt"), (3, 290, 77, "float16", "nn"), (33, 129, 84, "float32", "nt"),
          (40, 1001, 35, "float32", "nn"), (16, 16, 8, "float32", "nn")]
GPU = [(12, 1001, 1111, "bfloat16", "nn"), (12, 1001, 1111, "float16", "nt"), (128, 768, 3072, "float32", "nn"), (33, 1023, 777, "float32", "nt")]


def _case(m, n, k, dtype, layout):
    return dict(kind="matmul", m=m, n=n, k=k, dtype=dtype, layout=layout)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", SHAPES, ids=str)
@pytest.mark.parametrize("ahead", [8, 64])
def test_stays_in_bounds(c, ahead, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    it, launch = s.items[0], (C.c_int * 7)()
    source = _ffi.take_string(hiplib.poly_hip_render(it.root, b"k", 0, launch))
    assert "#define POLY_WAVES " in source
    source = source.replace("#define POLY_WAVES ", f"#define POLY_TOUCH_WGS {ahead}\n#define POLY_WAVES ", 1)
    sizes = [s.buf_slots[it.buf_slot_indices[p]].nbytes for p in range(it.n_buf_slots)]
    hostcheck.check_kernel(source, hostcheck._entry_name(source), (launch[0] + ahead, launch[1], launch[2]), launch[3], sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("c", GPU, ids=str)
def test_same_bits(c, monkeypatch):
    import torch
    state = cases.prepare(_case(*c), 7)
    assert "read B ahead" in state["plan"].kernel_info()[0]["desc"]
    got = cases.run(state)["C"]
    state["plan"].sync()
    monkeypatch.setenv("POLY_HIP_NO_PREFETCH", "1")
    plain = cases.prepare(_case(*c), 7)
    assert "read B ahead" not in plain["plan"].kernel_info()[0]["desc"]
    want = cases.run(plain)["C"]
    plain["plan"].sync()
    assert torch.equal(got, want)
