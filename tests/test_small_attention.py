"""kernels/attention_rows.hip: attention of few, ragged or fp32 queries and keys as one launch.
Queries and keys below, at and above the edges of its blocks (16 queries, units of 16 or 32
keys, one to eight waves, one and two query blocks to a workgroup), one key, the three operand
types.  Against softmax attention in float64 on the host, with the roundings of the unfused
kernels for 16-bit types (scores, masked scores, probabilities, output)."""
import ctypes as C
import math
import os
import sys

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

# batch, heads, queries = keys, type
SIZES = [(1, 12, 2, "bfloat16"), (1, 1, 3, "float32"), (3, 5, 12, "bfloat16"), (2, 3, 16, "float16"), (2, 3, 17, "float32"), (1, 3, 31, "float32"),
         (1, 4, 33, "bfloat16"), (2, 2, 64, "bfloat16"), (1, 2, 65, "float16"), (1, 3, 128, "bfloat16"), (1, 2, 130, "float32"), (1, 2, 257, "float32"),
         (2, 3, 345, "bfloat16"), (1, 2, 513, "bfloat16"), (1, 20, 840, "bfloat16"), (1, 2, 1024, "float32"), (1, 3, 1023, "float16")]


def _schedule(B, H, T, w):
    """The attention of a GPT-2 block over a fused q | k | v projection."""
    s, D = cases.Schedule(), 64 * H
    out, qkv, mask = s.buf("out", B * T * D, w), s.buf("qkv", 3 * B * T * D, w), s.buf("mask", T * T, w)

    def part(o):
        b, q, j = s.ranges(B, T, D)
        return s.store(s.tmp(B * T * D, w), b * (T * D) + q * D + j, qkv[b * (T * 3 * D) + q * (3 * D) + (j + o)], b, q, j)

    Q, K = part(0), part(D)
    b, e, q, n = s.ranges(B, H, T, T)
    k = s.rrange(64)
    at = b * (H * T * T) + e * (T * T) + q * T + n
    prod = Q[b * (T * D) + q * D + e * 64 + k].cast("float32") * K[b * (T * D) + n * D + e * 64 + k].cast("float32")
    sc = s.store(s.tmp(B * H * T * T, w), at, s.reduce("ADD", prod, k).cast(w), b, e, q, n)
    b, e, q, n = s.ranges(B, H, T, T)
    at = b * (H * T * T) + e * (T * T) + q * T + n
    sc = s.store(s.tmp(B * H * T * T, w), at, sc[at] * 0.125 + mask[q * T + n], b, e, q, n)

    def row(op, value):
        b, e, q = s.ranges(B, H, T)
        n = s.rrange(T)
        r = b * (H * T) + e * T + q
        return s.store(s.tmp(B * H * T), r, s.reduce(op, value(b * (H * T * T) + e * (T * T) + q * T + n, r), n), b, e, q)

    term = lambda a, r: ((sc[a].cast("float32") - top[r]) * cases.LOG2E).un("EXP2")  # noqa: E731
    top = row("MAX", lambda a, r: sc[a].cast("float32"))
    tot = row("ADD", term)
    b, e, q, n = s.ranges(B, H, T, T)
    at, r = b * (H * T * T) + e * (T * T) + q * T + n, b * (H * T) + e * T + q
    pr = s.store(s.tmp(B * H * T * T, w), at, (term(at, r) / tot[r]).cast(w), b, e, q, n)
    V = part(2 * D)
    b, e, q, j = s.ranges(B, H, T, 64)
    n = s.rrange(T)
    prod = pr[b * (H * T * T) + e * (T * T) + q * T + n].cast("float32") * V[b * (T * D) + n * D + e * 64 + j].cast("float32")
    s.store(out, b * (H * T * 64) + e * (T * 64) + q * 64 + j, s.reduce("ADD", prod, n).cast(w), b, e, q, j)
    return s


def _is_rows(text):
    return "attention_rows.hip" in text


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("B,H,T,w", SIZES)
def test_one_launch_in_bounds(B, H, T, w, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _schedule(B, H, T, w).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None) == 1
    src, n_items = C.c_void_p(), C.c_int()
    hiplib.poly_hip_fused_groups(pf.schedule, 0, C.byref(src), C.byref(n_items))
    text = _ffi.take_string(src.value)
    assert _is_rows(text) and n_items.value == s.n_items
    slots, launch = (C.c_int * 64)(), (C.c_int * 4)()
    n = hiplib.poly_hip_fused_group_launch(pf.schedule, 0, slots, 64, launch)
    sizes = [int(s.buf_slots[slots[i]].nbytes) for i in range(n)]
    threads = launch[0] * launch[3]
    hostcheck.check_kernel(text.split("\n// ---- ")[0], "poly_k", tuple(launch[:3]), launch[3], sizes, block_stride=max(1, threads >> 16))


@pytest.mark.gpu
@pytest.mark.parametrize("values", ["causal", "open", "first key only"])
@pytest.mark.parametrize("B,H,T,w", SIZES)
def test_against_float64(B, H, T, w, values):
    import torch
    D, dt = 64 * H, getattr(torch, w)
    g = torch.Generator().manual_seed(T)
    qkv = torch.randn(B, T, 3 * D, generator=g).to(dt)
    i = torch.arange(T)
    mask = dict(causal=torch.where(i[None, :] > i[:, None], -1e9 if w != "float16" else -6e4, 0.0), open=torch.randn(T, T, generator=g))
    mask = mask.get(values, torch.where(i[None, :].expand(T, T) > 0, float("-inf"), 0.0)).to(dt)
    plan = _schedule(B, H, T, w).plan()
    assert [k["klass"] for k in plan.kernel_info()] == ["attention-mfma"] and "scores of" in plan.kernel_info()[0]["desc"]
    data = [None] * len(plan.slots)
    by = {}
    for sl in plan.external_slots():
        v = dict(qkv=qkv, mask=mask).get(sl.name, torch.zeros(B * T * D, dtype=dt))
        data[sl.index] = by[sl.name] = v.cuda().reshape(-1)
    plan.run(data)
    got = by["out"].cpu().double().reshape(B, H, T, 64)
    rnd = lambda v: v.to(dt).double()  # noqa: E731
    q, k, v = (p.reshape(B, T, H, 64).permute(0, 2, 1, 3).double() for p in qkv.split(D, dim=2))
    x = rnd(rnd(rnd(q @ k.transpose(2, 3)) * 0.125) + mask.double())
    p = rnd(torch.softmax(x, 3))
    want = p @ v
    # 16-bit: a product on the other side of a rounding boundary moves a score by one step of
    # its type and all that follows by as much, relatively, as the largest score moves
    # (|x| <= 8 here: 2^-8 * 8 at most for one key, of which the row averages many), and the
    # output is rounded once.  fp32: 64 products and T terms of 2^-24 each, exp2 of arguments up to 2^4.
    eps = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 2.0 ** -23}[w]
    scale = (p @ v.abs())
    bound = scale * (eps * 8 if w != "float32" else eps * (64 + math.sqrt(T))) + 1e-30
    err = (got - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    if values == "first key only":
        assert torch.equal(got, v[:, :, :1].expand(B, H, T, 64))
