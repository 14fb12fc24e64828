"""Products on kernels/matmul_wave.hip are no less exact than on the template that has them
with POLY_HIP_NO_WAVE_MM=1: an output is the sum of no fewer partial sums, and its error
against float64 no larger.  Depths from 2048 on, where the fp32 tile template deals the depth
to four, five, six and seven workgroups, and shallower ones, where it does not."""
import ctypes as C
import re

import pytest

from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, _name, cases

DEEP = [(80, 1096, 2304, "nn"), (80, 152, 2048, "nt"), (104, 1424, 2560, "nn"), (128, 768, 3072, "nn"), (345, 768, 3072, "nn"), (400, 2728, 3840, "nn"),
        (632, 328, 3840, "nt"), (1464, 440, 3584, "nt"), (2464, 152, 2048, "tn")]
OTHER = [(128, 768, 768, "nn"), (300, 64, 2048, "nn"), (64, 704, 4096, "tn")]


def _partial_sums(text):
    def number(pattern, default=1):
        m = re.search(pattern, text)
        return int(m.group(1)) if m else default
    return number(r"depth dealt to (\d+) waves") * (2 if "of two sums each" in text else 1) * number(r"K dealt to (\d+) workgroups")


@pytest.mark.parametrize("c", DEEP + OTHER, ids=_name)
def test_no_fewer_partial_sums(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    m, n, k, layout = c
    pf = cases._matmul_schedule(_case(m, n, k, "float32", layout)).plan()
    root = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents.items[0].root
    here = _ffi.take_string(hiplib.poly_hip_describe(root, 0))
    monkeypatch.setenv("POLY_HIP_NO_WAVE_MM", "1")
    there = _ffi.take_string(hiplib.poly_hip_describe(root, 0))
    assert "depth dealt to" in here and "32x32x2 f32" in there
    assert ("K dealt to" in there) == (c in DEEP)
    assert _partial_sums(here) >= _partial_sums(there), (here, there)


@pytest.mark.gpu
@pytest.mark.parametrize("c", DEEP + OTHER, ids=_name)
def test_error_against_float64_is_no_larger(c, monkeypatch):
    m, n, k, layout = c
    case = _case(m, n, k, "float32", layout)

    def error():
        state = cases.prepare(case, 5)
        got = cases.run(state)["C"]
        state["plan"].sync()
        by = {s.name: state["data"][s.index].double() for s in state["plan"].external_slots()}
        a = by["A"].reshape(k, m).T if layout[0] == "t" else by["A"].reshape(m, k)
        b = by["B"].reshape(n, k).T if layout[1] == "t" else by["B"].reshape(k, n)
        want = a @ b
        return float((got.double().reshape(m, n) - want).norm() / want.norm())

    here = error()
    monkeypatch.setenv("POLY_HIP_NO_WAVE_MM", "1")
    there = error()
    # both are averages over more than 10000 elements: 1 % for the two samples
    assert here <= 1.01 * there, (here, there)
