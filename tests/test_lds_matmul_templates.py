"""The 16-bit templates that stage tiles in LDS (kernels/matmul_dma.hip and
kernels/matmul_mfma.hip) at the sizes of few tiles, which kernels/matmul_wave.hip and the 64-row
tiles take unless switched off, and on narrow outputs of many tiles, which reach the 64-wide
register-staged form by dispatch.  Ragged rows and columns and every layout of the operands;
each case says which template it is about.  Against the product in float64 within the
rounding of K fp32 additions (the products of 16-bit values are exact)."""
import ctypes as C
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_small_matmul import _case, _name, cases

NO_SMALL = ("POLY_HIP_NO_WAVE_MM", "POLY_HIP_NO_SMALL_TILES")
STAGED = NO_SMALL + ("POLY_HIP_NO_DMA",)
FEW = [(256, 512, 128, "bfloat16", "nn"), (256, 512, 128, "bfloat16", "nt"), (128, 192, 64, "bfloat16", "nn"), (200, 328, 192, "bfloat16", "nt"), (136, 128, 64, "float16", "tn")]
NARROW = [(64, 4160, 128, "bfloat16", "nn"), (4160, 64, 128, "bfloat16", "nn"), (63, 4168, 192, "bfloat16", "nn"), (4161, 64, 128, "bfloat16", "nt"), (4168, 56, 128, "float16", "tn")]
# case, switches, what its description says, whether its operands go straight into LDS
ALL = ([(c, NO_SMALL, "tile 128x128x64", True) for c in FEW] + [(c, STAGED, "tile 128x128x64", False) for c in FEW] +
       [((64, 1000, 64, "bfloat16", "nt"), NO_SMALL, "tile 64x256x64", False)] +
       [(c, (), "tile 64x256x64" if c[0] <= 64 else "tile 256x64x64", False) for c in NARROW])


def _id(v):
    return _name(v) if len(v) == 5 else "staged" if v == STAGED else "no-small" if v else "as-dispatched"


@pytest.fixture
def switched(monkeypatch):
    def on(switches):
        for s in switches:
            monkeypatch.setenv(s, "1")
    return on


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c,switches,tile,direct", [pytest.param(*a, id=f"{_name(a[0])}-{_id(a[1])}") for a in ALL])
def test_stays_in_bounds(c, switches, tile, direct, hiplib, monkeypatch, switched):
    switched(switches)
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    desc = _ffi.take_string(hiplib.poly_hip_describe(s.items[0].root, 0))
    assert tile in desc and ("straight into LDS" in desc) == direct, desc
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c,switches,tile,direct", [pytest.param(*a, id=f"{_name(a[0])}-{_id(a[1])}") for a in ALL])
def test_against_float64(c, switches, tile, direct, switched):
    import torch
    switched(switches)
    m, n, k, dtype, layout = c
    state = cases.prepare(_case(*c), 5)
    desc = state["plan"].kernel_info()[0]["desc"]
    assert tile in desc and ("straight into LDS" in desc) == direct, desc
    got = cases.run(state)["C"]
    state["plan"].sync()
    by_name = {s.name: state["data"][s.index] for s in state["plan"].external_slots()}
    a, b = by_name["A"].double().cpu(), by_name["B"].double().cpu()
    a = a.reshape(k, m).T if layout[0] == "t" else a.reshape(m, k)
    b = b.reshape(n, k).T if layout[1] == "t" else b.reshape(k, n)
    err = (got.double().cpu().reshape(m, n) - a @ b).abs()
    bound = k * 2.0 ** -24 * (a.abs() @ b.abs())
    assert bool((err <= bound).all()), float((err / bound).max())
    state["plan"].close()
