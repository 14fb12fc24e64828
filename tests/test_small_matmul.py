"""Products of few or ragged output tiles.  kernels/matmul_wave.hip: every extent at, below
and above the edges of its tiles, the depth below one step, at whole steps of all waves and
with a remainder, operands along the depth and along their rows, the three input types.
kernels/matmul_dma.hip on tiles of 64 rows: ragged rows and columns, a depth of the fewest
and of many K tiles, every layout, two, three, four and six stages.
Against the product in float64, element by element, within the rounding of K fp32 additions
and products (K * 2^-24 * sum of |a b|; the products of 16-bit values are exact)."""
import ctypes as C
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

EDGES = [(12, 33, 8, "bfloat16", "nn"), (16, 32, 256, "bfloat16", "nn"), (17, 31, 255, "bfloat16", "nt"), (12, 770, 1000, "bfloat16", "nn"),
         (65, 63, 777, "bfloat16", "tn"), (37, 1280, 291, "float16", "nn"), (333, 219, 188, "bfloat16", "nn"), (900, 1410, 70, "bfloat16", "tn"),
         (1500, 1283, 101, "bfloat16", "nt"), (2, 5, 9, "float32", "nn"), (15, 16, 128, "float32", "nt"), (143, 40, 791, "float32", "nn"),
         (33, 129, 784, "float32", "nt"), (200, 50, 4096, "float32", "tn"), (64, 700, 5000, "float32", "nn"), (200, 300, 4095, "float32", "tn"), (130, 770, 515, "float32", "nn"), (17, 96, 9000, "bfloat16", "nn"), (64, 96, 4100, "float32", "nn"), (600, 650, 67, "float32", "nt")]

LDS_TILES = [(333, 840, 256, "bfloat16", "nn", "64x64x64"), (345, 768, 3072, "bfloat16", "nn", "64x64x64"), (1000, 904, 256, "bfloat16", "nt", "64x64x64"),
             (1000, 904, 320, "float16", "tn", "64x64x64"), (1111, 1000, 1536, "bfloat16", "nt", "64x128x64"), (1112, 1000, 256, "bfloat16", "tn", "64x128x64"),
             (1035, 3000, 768, "bfloat16", "nn", "64x128x64")]
ALL = [(c, "depth dealt to") for c in EDGES] + [(c[:5], "tile " + c[5]) for c in LDS_TILES]


def _name(c):
    return "-".join(str(v) for v in c)


def _case(m, n, k, dtype, layout):
    return dict(kind="matmul", m=m, n=n, k=k, dtype=dtype, layout=layout)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c,how", ALL, ids=lambda v: _name(v) if isinstance(v, tuple) else "")
def test_stays_in_bounds(c, how, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert how in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c,how", ALL, ids=lambda v: _name(v) if isinstance(v, tuple) else "")
def test_against_float64(c, how):
    import torch
    m, n, k, dtype, layout = c
    state = cases.prepare(_case(*c), 5)
    assert how in state["plan"].kernel_info()[0]["desc"]
    got = cases.run(state)["C"]
    state["plan"].sync()
    by_name = {s.name: state["data"][s.index] for s in state["plan"].external_slots()}
    a, b = by_name["A"].double().cpu(), by_name["B"].double().cpu()
    a = a.reshape(k, m).T if layout[0] == "t" else a.reshape(m, k)
    b = b.reshape(n, k).T if layout[1] == "t" else b.reshape(k, n)
    err = (got.double().cpu().reshape(m, n) - a @ b).abs()
    bound = k * 2.0 ** -24 * (a.abs() @ b.abs())
    assert bool((err <= bound).all()), float((err / bound).max())
    assert torch.isfinite(got).all()
