"""fp32 products of a depth of 4096 and more on more than 64 rows and columns (the 32x32 blocks of
kernels/matmul_wave.hip): extents at, below and above the edges of a 64x64 tile, a depth of whole
steps and with a remainder, dealt to one, two, eight and sixteen workgroups, every layout.
Against the product in float64, element by element, within the rounding of K fp32 additions
and products (K * 2^-24 * sum of |a b|), and the error no larger than the tile template's."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, _name, cases

DEEP = [(65, 65, 4096, "nn", 8), (128, 66, 4100, "nt", 1), (129, 191, 4097, "tn", 1), (512, 784, 4096, "tn", 2), (384, 900, 4128, "nn", 2), (70, 130, 8192, "nn", 16), (192, 193, 5000, "nt", 2),
        (700, 700, 4112, "tn", 2), (1000, 1024, 4104, "nn", 1), (829, 863, 18832, "tn", 1)]


def _form(split):
    return "K dealt to %d workgroups per tile" % split if split > 1 else "depth dealt to 4 waves of two sums each"


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", DEEP[:7], ids=_name)
def test_stays_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c[:3], "float32", c[3])).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    desc = _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert "mfma 32x32x2 f32" in desc and "depth dealt to 4 waves" in desc and _form(c[4]) in desc
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.parametrize("m,n,k,layout,here", [(344, 136, 21424, "tn", False), (344, 136, 21504, "tn", True), (910, 1108, 12960, "nt", False), (910, 1108, 12961, "nt", True),
                                               (466, 524, 15648, "nt", False), (466, 524, 15360, "nt", True), (126, 108, 15840, "nt", True), (147, 315, 5808, "nn", True),
                                               (829, 863, 18832, "tn", True)])
def test_which_template(m, n, k, layout, here, hiplib, monkeypatch):
    """A depth that 16 and 32 do not divide well goes to the tile template where that deals it to several times
    as many workgroups; one that it cannot deal at all, or rows that it cannot read, stay."""
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(m, n, k, "float32", layout)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert ("depth dealt to" in _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))) == here


@pytest.mark.gpu
@pytest.mark.parametrize("c", DEEP, ids=_name)
def test_against_float64(c, monkeypatch):
    import torch
    m, n, k, layout, split = c

    def error():
        state = cases.prepare(_case(m, n, k, "float32", layout), 8)
        desc = state["plan"].kernel_info()[0]["desc"]
        got = cases.run(state)["C"]
        state["plan"].sync()
        by = {s.name: state["data"][s.index].double().cpu() for s in state["plan"].external_slots()}
        a = by["A"].reshape(k, m).T if layout[0] == "t" else by["A"].reshape(m, k)
        b = by["B"].reshape(n, k).T if layout[1] == "t" else by["B"].reshape(k, n)
        want = a @ b
        err = (got.double().cpu().reshape(m, n) - want).abs()
        assert bool((err <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all())
        return float(err.norm() / want.norm()), desc

    here, desc = error()
    assert _form(split) in desc
    monkeypatch.setenv("POLY_HIP_NO_WAVE_MM", "1")
    there, desc = error()
    assert "depth dealt" not in desc
    # (two orders of the same roundings: the errors of two runs of one order on other inputs differ by a few percent)
    assert here <= 1.1 * there, (here, there)
