"""kernels/attention_rows.hip beyond equal queries and keys: more of either than of the other,
two blocks of 16 queries to a workgroup for every type, and terms too small for a normal
float.  Against softmax attention in float64 on the host with the roundings of the unfused
kernels for 16-bit types."""
import ctypes as C
import math
import os

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi
from test_small_attention import _is_rows, cases

# batch, heads, queries, keys, type
SIZES = [(1, 2, 5, 300, "bfloat16"), (2, 3, 300, 5, "bfloat16"), (1, 3, 700, 17, "float32"), (1, 4, 16, 1024, "float16"), (2, 2, 33, 1000, "float32"),
         (1, 2, 129, 64, "float16"), (1, 2, 128, 72, "bfloat16")]
TWO_BLOCKS = [(1, 16, 1023, 1023, "float32"), (1, 18, 930, 70, "float16"), (2, 16, 500, 33, "bfloat16")]


def _name(c):
    return "-".join(str(v) for v in c)


def _schedule(B, H, M, N, w):
    s, D, F32 = cases.Schedule(), 64 * H, "float32"
    out, Q, K, V, mask = s.buf("out", B * M * D, w), s.buf("q", B * M * D, w), s.buf("k", B * N * D, w), s.buf("v", B * N * D, w), s.buf("mask", M * N, w)

    def scores():
        b, e, q, n = s.ranges(B, H, M, N)
        return (b, e, q, n), b * (H * M * N) + e * (M * N) + q * N + n

    rs, at = scores()
    b, e, q, n = rs
    k = s.rrange(64)
    prod = Q[b * (M * D) + q * D + e * 64 + k].cast(F32) * K[b * (N * D) + n * D + e * 64 + k].cast(F32)
    sc = s.store(s.tmp(B * H * M * N, w), at, s.reduce("ADD", prod, k).cast(w), *rs)
    rs, at = scores()
    sc = s.store(s.tmp(B * H * M * N, w), at, sc[at] * 0.125 + mask[rs[2] * N + rs[3]], *rs)

    def row(op, value):
        b, e, q = s.ranges(B, H, M)
        n = s.rrange(N)
        r = b * (H * M) + e * M + q
        return s.store(s.tmp(B * H * M), r, s.reduce(op, value(b * (H * M * N) + e * (M * N) + q * N + n, r), n), b, e, q)

    term = lambda a, r: ((sc[a].cast(F32) - top[r]) * cases.LOG2E).un("EXP2")  # noqa: E731
    top = row("MAX", lambda a, r: sc[a].cast(F32))
    tot = row("ADD", term)
    rs, at = scores()
    r = rs[0] * (H * M) + rs[1] * M + rs[2]
    pr = s.store(s.tmp(B * H * M * N, w), at, (term(at, r) / tot[r]).cast(w), *rs)
    b, e, q, j = s.ranges(B, H, M, 64)
    n = s.rrange(N)
    prod = pr[b * (H * M * N) + e * (M * N) + q * N + n].cast(F32) * V[b * (N * D) + n * D + e * 64 + j].cast(F32)
    s.store(out, b * (H * M * 64) + e * (M * 64) + q * 64 + j, s.reduce("ADD", prod, n).cast(w), b, e, q, j)
    return s


def _rendered(hiplib, monkeypatch, c):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = _schedule(*c).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    assert hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None) == 1
    src, n_items = C.c_void_p(), C.c_int()
    hiplib.poly_hip_fused_groups(pf.schedule, 0, C.byref(src), C.byref(n_items))
    text = _ffi.take_string(src.value)
    assert _is_rows(text) and n_items.value == s.n_items
    return pf, s, text.split("\n// ---- ")[0]


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", SIZES + TWO_BLOCKS, ids=_name)
def test_one_launch_in_bounds(c, hiplib, monkeypatch):
    pf, s, text = _rendered(hiplib, monkeypatch, c)
    assert f"#define POLY_FA_QT {2 if c in TWO_BLOCKS else 1}\n" in text
    slots, launch = (C.c_int * 64)(), (C.c_int * 4)()
    n = hiplib.poly_hip_fused_group_launch(pf.schedule, 0, slots, 64, launch)
    sizes = [int(s.buf_slots[slots[i]].nbytes) for i in range(n)]
    hostcheck.check_kernel(text, "poly_k", tuple(launch[:3]), launch[3], sizes, block_stride=max(1, launch[0] * launch[3] >> 16))


@pytest.mark.parametrize("c", [(1, 2, 5, 300, "bfloat16"), (1, 3, 700, 17, "float32")], ids=_name)
def test_terms_as_the_unfused_kernels_compute_them(c, hiplib, monkeypatch):
    """Shapes that no other fused form takes, types with probabilities below 2^-126: the exp2 of
    the unfused kernels, which reaches them (the bare instruction gives 0 there)."""
    _, _, text = _rendered(hiplib, monkeypatch, c)
    generated = text[:text.index("// attention_rows.hip")]
    assert "__builtin_exp2f(" in generated and "__builtin_amdgcn_exp2f(" not in generated


def _run(c, q, k, v, mask):
    B, H, M, N, w = c
    plan = _schedule(*c).plan()
    assert [i["klass"] for i in plan.kernel_info()] == ["attention-mfma"] and "scores of" in plan.kernel_info()[0]["desc"]
    import torch
    data, by = [None] * len(plan.slots), {}
    for sl in plan.external_slots():
        t = dict(q=q, k=k, v=v, mask=mask).get(sl.name, torch.zeros(B * M * 64 * H, dtype=getattr(torch, w)))
        data[sl.index] = by[sl.name] = t.cuda().reshape(-1)
    plan.run(data)
    return by["out"].cpu().double().reshape(B, H, M, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("masked", ["causal", "open"])
@pytest.mark.parametrize("c", SIZES + TWO_BLOCKS, ids=_name)
def test_against_float64(c, masked):
    import torch
    B, H, M, N, w = c
    D, dt = 64 * H, getattr(torch, w)
    g = torch.Generator().manual_seed(M + N)
    q, k, v = (torch.randn(B, n, D, generator=g).to(dt) for n in (M, N, N))
    # (at least the first key is seen by every query)
    later = torch.arange(N)[None, :] > torch.arange(M)[:, None]
    mask = (torch.where(later, -1e9 if w != "float16" else -6e4, 0.0) if masked == "causal" else torch.randn(M, N, generator=g)).to(dt)
    got = _run(c, q, k, v, mask)
    rnd = lambda t: t.to(dt).double()  # noqa: E731
    qh, kh, vh = (t.reshape(B, -1, H, 64).permute(0, 2, 1, 3).double() for t in (q, k, v))
    x = rnd(rnd(rnd(qh @ kh.transpose(2, 3)) * 0.125) + mask.double())
    p = rnd(torch.softmax(x, 3))
    # 16-bit: a score on the other side of a rounding boundary moves its term by one step of its
    # type times the largest score (|x| <= 8); the output is rounded once.  fp32: 64 products
    # and N terms of 2^-24 each, exp2 of arguments up to 2^4.
    eps = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 2.0 ** -23}[w]
    bound = (p @ vh.abs()) * (eps * 8 if w != "float32" else eps * (64 + math.sqrt(N))) + 1e-30
    err = (got - p @ vh).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(1, 2, 7, 40, "bfloat16"), (1, 2, 7, 40, "float32"), (1, 16, 1023, 40, "bfloat16")], ids=_name)
def test_probabilities_below_the_normal_floats(c):
    """Scores 87.5 to 90 below the row's largest: terms and probabilities of 2^-126.2 to 2^-129.8
    under values of 2^110, the largest score's value being 0."""
    import torch
    B, H, M, N, w = c
    D, dt = 64 * H, getattr(torch, w)
    q, k = torch.zeros(B, M, D, dtype=dt), torch.zeros(B, N, D, dtype=dt)
    v = torch.full((B, N, D), 2.0 ** 110)
    v[:, 0] = 0.0
    mask = torch.tensor([0.0] + [(-87.5, -88.0, -88.5, -89.0, -90.0)[n % 5] for n in range(1, N)]).expand(M, N).contiguous()
    got = _run(c, q, k, v.to(dt), mask.to(dt))
    p = torch.exp2((mask[0].double() * cases.LOG2E))[1:]
    want = float(p.sum()) * 2.0 ** 110
    # a probability is a multiple of 2^-133 (bf16) or 2^-149 (fp32), half a step off at most in
    # the term, in the quotient and in its rounding; the arguments of exp2 carry 2^-17; the output 2^-8 (bf16) or N additions
    step = 2.0 ** -133 if w == "bfloat16" else 2.0 ** -149
    bound = (N * step * 1.5 * 2.0 ** 110) + want * (2.0 ** -16 + (2.0 ** -8 if w == "bfloat16" else N * 2.0 ** -24))
    assert float((got - want).abs().max()) <= bound < want / 4, (float(got.min()), float(got.max()), want, bound)


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(1, 2, 70, 100, "bfloat16"), (1, 2, 70, 100, "float16"), (1, 2, 70, 100, "float32"), (1, 16, 1023, 40, "bfloat16")], ids=_name)
def test_non_finite_rows_and_values(c):
    """Where a fused unit of keys has no terms but zeros, its values still meet them: an infinite value
    under a masked key gives NaN as 0 * inf does; a row without any key, and one with a NaN score, are NaN
    as a whole; rows beside them are what they are without these."""
    import torch
    B, H, M, N, w = c
    D, dt = 64 * H, getattr(torch, w)
    g = torch.Generator().manual_seed(N)
    q, k, v = (torch.randn(B, n, D, generator=g).to(dt) for n in (M, N, N))
    mask = torch.where(torch.arange(N)[None, :] > torch.arange(M)[:, None] % N, -6e4, 0.0)
    clean = _run(c, q, k, v, mask.to(dt))
    mask[3], mask[20, 5] = -math.inf, math.nan
    v[:, N - 1, 7] = math.inf                    # of head 0: under a masked key for all but the rows that see it
    got = _run(c, q, k, v, mask.to(dt))
    assert bool(got[:, :, [3, 20]].isnan().all())
    rows = [m for m in range(M) if m not in (3, 20)]
    masked = [m for m in rows if m % N < N - 1]
    assert bool(got[:, 0, masked, 7].isnan().all())
    got, clean = got[:, :, rows].clone(), clean[:, :, rows].clone()
    got[:, 0, :, 7] = clean[:, 0, :, 7] = 0.0
    assert bool((got == clean).all())
