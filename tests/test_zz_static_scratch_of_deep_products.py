"""Deep 16-bit products through the descriptor row and the entry point that allocates nothing: a product
whose plan form leaves 64 MiB of partial sums is lowered to one that fits the 32 MiB of the static array, at
that size exactly and just under it.  The bits of poly_hip_execute, and the product in float64 within the
rounding of K fp32 additions."""
import ctypes as C
import os
import sys

import pytest

from polygrad_amd import PlanFile, _ffi
from test_deep_16bit_products import _case

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [(2048, 2048, 16384, "bfloat16", "nt"), (1960, 2040, 16384, "float16", "tn")], ids=str)
def test_deep_product_on_the_static_array(c, monkeypatch):
    import torch
    m, n, k, dtype, layout = c
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(*c)).plan()
    sched = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    lib = _ffi.load()
    assert lib.poly_hip_init() == 0
    desc = lib.poly_hip_backend_desc().contents
    runner = _ffi.PolyRunner()
    assert desc.lower_item(None, sched.items[0].root, b"deep", C.byref(runner)) == 0
    g = torch.Generator(device="cuda").manual_seed(k)
    by = dict(A=torch.randn(m * k, generator=g, device="cuda").to(getattr(torch, dtype)), B=torch.randn(n * k, generator=g, device="cuda").to(getattr(torch, dtype)))
    outs = []
    try:
        for fn in (lib.poly_hip_execute_static, lib.poly_hip_execute):
            by["C"] = torch.zeros(m * n, device="cuda")
            torch.cuda.synchronize()
            item = sched.items[0]
            args = (C.c_void_p * item.n_buf_slots)(*[by[pf.names[item.buf_slot_indices[j]]].data_ptr() for j in range(item.n_buf_slots)])
            assert fn(C.byref(runner), args, item.n_buf_slots) == 0
            assert lib.poly_hip_sync() == 0
            outs.append(by["C"])
    finally:
        desc.free_runner(C.byref(runner))
    assert torch.equal(outs[0], outs[1])
    a = by["A"].double().reshape(k, m).T if layout[0] == "t" else by["A"].double().reshape(m, k)
    b = by["B"].double().reshape(n, k).T if layout[1] == "t" else by["B"].double().reshape(k, n)
    err = (outs[0].double().reshape(m, n) - a @ b).abs()
    assert bool((err <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all())
