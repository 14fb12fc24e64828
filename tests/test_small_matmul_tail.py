"""kernels/matmul_wave.hip with an epilogue: bias, an activation, and the value between them
stored too, because a later kernel reads it (a layer's pre-activation, kept for its backward
pass).  Depths that one workgroup has and depths dealt to several, whose sums a second kernel
adds up and finishes; both thin sides; a batch range; rows and depth of two digits each (the
projection behind attention reads its heads where they lie)."""
import ctypes as C
import os
import re
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

# rows, columns, depth, type, form, workgroups that share a tile's depth
CASES = [(32, 512, 2048, "float32", "plain", 1), (32, 512, 4096, "float32", "plain", 4), (32, 512, 4100, "float32", "plain", 1), (32, 512, 8192, "float32", "plain", 4),
         (300, 64, 2048, "float32", "plain", 1), (300, 64, 4096, "float32", "plain", 4), (300, 64, 4104, "float32", "plain", 2), (300, 10, 8192, "float32", "plain", 8),
         (33, 72, 130, "float32", "batch", 1), (20, 40, 4096, "float32", "batch", 8), (36, 130, 192, "float32", "heads", 1), (60, 24, 4096, "float32", "heads", 8),
         (12, 776, 520, "bfloat16", "plain", 1), (63, 264, 1001, "float16", "plain", 1), (33, 72, 130, "bfloat16", "batch", 1), (36, 136, 192, "bfloat16", "heads", 1)]
BATCH = dict(plain=1, batch=3, heads=1)


def _name(c):
    return "-".join(str(v) for v in c)


def _schedule(M, N, K, w, form):
    """pre = A B + bias; out = pre (1 + pre); kept = 2 pre, of which only pre is an intermediate."""
    s, Z = cases.Schedule(), BATCH[form]
    out, kept = s.buf("out", Z * M * N, w), s.buf("kept", Z * M * N, w)
    A, B, bias = s.buf("A", Z * M * K, w), s.buf("B", Z * K * N, w), s.buf("bias", N, w)
    T = M // 3

    def ranges():
        if form == "heads":
            b, q, j = s.ranges(3, T, N)
            return (b, q, j), b * (T * N) + q * N + j
        if form == "batch":
            z, m, j = s.ranges(Z, M, N)
            return (z, m, j), z * (M * N) + m * N + j
        m, j = s.ranges(M, N)
        return (m, j), m * N + j

    rs, at = ranges()
    k = s.rrange(K)
    j = rs[-1]
    if form == "heads":
        a, b = rs[0] * (T * K) + (k // 64) * (T * 64) + rs[1] * 64 + k % 64, k * N + j
    elif form == "batch":
        a, b = rs[0] * (M * K) + rs[1] * K + k, rs[0] * (K * N) + k * N + j
    else:
        a, b = rs[0] * K + k, k * N + j
    acc = s.reduce("ADD", A[a].cast("float32") * B[b].cast("float32"), k).cast(w)
    pre = s.store(s.tmp(Z * M * N, w), at, acc + bias[j], *rs)
    rs, at = ranges()
    s.store(out, at, pre[at] * (1.0 + pre[at]), *rs)
    rs, at = ranges()
    s.store(kept, at, 2.0 * pre[at], *rs)
    return s


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", CASES, ids=_name)
def test_value_between_is_stored_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _schedule(*c[:5]).plan()
    assert hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None) >= 1
    src, n_items = C.c_void_p(), C.c_int()
    hiplib.poly_hip_fused_groups(pf.schedule, 0, C.byref(src), C.byref(n_items))
    text = _ffi.take_string(src.value)
    assert n_items.value == 2 and "matmul_wave.hip" in text
    # by the kernel that has the whole sum, and by no other
    finishing, *stages = text.split("\n// ---- first stage")
    assert len(stages) == (c[5] > 1) and re.search(r"#define POLY_KSPLIT (\d+)", finishing).group(1) == str(c[5])
    assert finishing.count("#define POLY_EP_MID_VALUE") == 1 and "*POLY_EP_MID_PTR(m, n, z) = POLY_EP_MID_VALUE(" in finishing
    assert not any("#define POLY_EP_MID_VALUE" in st for st in stages)
    assert hostcheck.check_schedule(hiplib, pf.schedule) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=_name)
def test_both_buffers_against_float64(c):
    import torch
    M, N, K, w, form, _ = c
    Z, dt = BATCH[form], getattr(torch, w)
    plan = _schedule(M, N, K, w, form).plan()
    desc = [k["desc"] for k in plan.kernel_info()]
    assert any("depth dealt to" in d and "a value on the way stored as well" in d for d in desc), desc
    g = torch.Generator().manual_seed(K)
    x, y, b = (torch.randn(n, generator=g) for n in (Z * M * K, Z * K * N, N))
    host = dict(A=x.to(dt), B=(y / K ** 0.5).to(dt), bias=b.to(dt))
    data, by = [None] * len(plan.slots), {}
    for sl in plan.external_slots():
        data[sl.index] = by[sl.name] = host.get(sl.name, torch.full((Z * M * N,), float("nan"), dtype=dt)).cuda()
    for _ in range(3):
        plan.run(data)
    a = host["A"].double()
    a = a.reshape(3, K // 64, M // 3, 64).permute(0, 2, 1, 3).reshape(1, M, K) if form == "heads" else a.reshape(Z, M, K)
    bm, bias = host["B"].double().reshape(Z, K, N), host["bias"].double()
    want, size = a @ bm + bias, a.abs() @ bm.abs()
    pre = by["kept"].cpu() / 2                      # (exact)
    # K fp32 additions and products, the bias, and for 16-bit types a rounding of the sum and one of the result
    step = {"float32": 2.0 ** -24, "bfloat16": 2.0 ** -8, "float16": 2.0 ** -11}[w]
    bound = K * 2.0 ** -24 * size + step * (2 * want.abs() + bias.abs()) + step * K * 2.0 ** -24 * size
    err = (pre.double().reshape(Z, M, N) - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    # and the activation of that very value, a rounding per operation
    assert torch.equal(by["out"].cpu(), pre * (1.0 + pre))
    plan.close()
