"""Kernels that copy a whole buffer cost no launch: readers of an intermediate copy read what it
copies, and what is copied into a buffer of the caller's is written there by the kernel that makes
it.  Which copies go, and the same bits as with all of them launched -- also where buffers of the
caller share memory, when a buffer written early would be read late."""
import os
import sys

import pytest

from polygrad_amd import PlanFile

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

N, K = 40, 300


def s_i(s):
    """The first range of the kernel that is being put together."""
    return cases.E("RANGE", "int32", (cases.const(N),), (0, 3), N)


def _copy(s, dst, src):
    (i,) = s.ranges(src.numel)
    return s.store(dst, i, src[i], i)


def _sums(s, x, dst, value=lambda v: v):
    (i,) = s.ranges(N)
    k = s.rrange(K)
    return s.store(dst, i, value(s.reduce("ADD", x[i * K + k], k)), i)


def _scaled(s, x, dst, by, at=lambda i: i):
    (i,) = s.ranges(N)
    return s.store(dst, i, x[at(i)] * by, i)


def _schedule(what):
    """(schedule, copies that need no launch)"""
    s = cases.Schedule()
    x, p, out = s.buf("x", N * K), s.buf("p", N), s.buf("out", N)
    if what == "intermediate":
        c = _copy(s, s.tmp(N), _sums(s, x, s.tmp(N)))
        _sums(s, x, out, lambda v: v + c[s_i(s) * -1 + (N - 1)])
        return s, 1
    if what == "copy of a copy":
        c = _copy(s, s.tmp(N), _copy(s, s.tmp(N), _sums(s, x, s.tmp(N))))
        _sums(s, x, out, lambda v: v + c[s_i(s) * -1 + (N - 1)])
        return s, 2
    if what == "update in place":
        (i,) = s.ranges(N)
        k = s.rrange(K)
        new = s.store(s.tmp(N), i, p[i] - s.reduce("ADD", x[i * K + k], k) * 0.01, i)
        _copy(s, p, new)
        _sums(s, x, out, lambda v: v + p[s_i(s) * -1 + (N - 1)])
        return s, 1
    if what == "update reads other elements":
        (i,) = s.ranges(N)
        k = s.rrange(K)
        new = s.store(s.tmp(N), i, p[i * -1 + (N - 1)] - s.reduce("ADD", x[i * K + k], k) * 0.01, i)
        _copy(s, p, new)
        return s, 0
    if what == "old value read behind the update":
        (i,) = s.ranges(N)
        k = s.rrange(K)
        new = s.store(s.tmp(N), i, p[i] - s.reduce("ADD", x[i * K + k], k) * 0.01, i)
        _sums(s, x, out, lambda v: v + p[s_i(s) * -1 + (N - 1)])
        _copy(s, p, new)
        return s, 0
    if what == "copied in another order":
        t = _sums(s, x, s.tmp(N))
        c = _scaled(s, t, s.tmp(N), 1.0, lambda i: i * -1 + (N - 1))
        _sums(s, x, out, lambda v: v + c[s_i(s)])
        return s, 0
    if what == "part of a buffer":
        t = _sums(s, x, s.tmp(N))
        c = s.tmp(N)
        (i,) = s.ranges(N // 2)
        s.store(c, i, t[i], i)
        _sums(s, x, out, lambda v: v + c[s_i(s) * -1 + (N - 1)])
        return s, 0
    if what == "written twice":
        t = _sums(s, x, s.tmp(N))
        c = _copy(s, s.tmp(N), t)
        _sums(s, x, t, lambda v: v * 2.0)
        _sums(s, x, out, lambda v: v + c[s_i(s) * -1 + (N - 1)])
        return s, 0
    assert what == "copy of an input"
    c = _copy(s, s.tmp(N), p)
    _sums(s, x, out, lambda v: v + c[s_i(s) * -1 + (N - 1)])
    return s, 0


WHAT = ["intermediate", "copy of a copy", "update in place", "update reads other elements", "old value read behind the update", "copied in another order", "part of a buffer",
        "written twice", "copy of an input"]


@pytest.mark.parametrize("what", WHAT)
def test_which_copies_go(what, hiplib, monkeypatch, capfd):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    monkeypatch.setenv("POLY_HIP_DEBUG", "1")
    s, n = _schedule(what)
    assert hiplib.poly_hip_fused_groups(s.plan().schedule, -1, None, None) >= 0
    said = [line for line in capfd.readouterr().err.splitlines() if "need no launch" in line]
    assert [int(line.split(": ")[2].split()[0]) for line in said] == ([n] if n else [])


def test_groups_are_refined_once(hiplib, monkeypatch, capfd):
    """Which copies go is found out with the groups as they are first; those that work in pairs (attention and
    the product its keys come from, one in each of 12 layers) are rendered for each other once."""
    monkeypatch.setenv("POLY_HIP_DEBUG", "1")
    pf = PlanFile(os.path.join(cases.PLANS, "gpt2_small_bf16_b8_t1024.polyplan"))
    assert hiplib.poly_hip_fused_groups(pf.schedule, -1, None, None) > 12
    err = capfd.readouterr().err
    assert err.count("leaves the block maxima of the keys") == 12 and err.count("need no launch") == 1


def _run(plan, shared):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    data, by = [None] * len(plan.slots), {}
    for slot in plan.external_slots():
        by[slot.name] = data[slot.index] = torch.rand(slot.numel, generator=g, device="cuda")
    for small, large in shared:         # one buffer at the start of another
        index = [s.index for s in plan.external_slots() if s.name == small][0]
        data[index] = by[small] = by[large][:by[small].numel()]
    for _ in range(3):
        plan.run(data)
    return {k: v.cpu().numpy().tobytes() for k, v in by.items()}, len(plan.kernel_info())


@pytest.mark.gpu
@pytest.mark.parametrize("what", WHAT)
def test_same_bits_as_with_the_copies(what, monkeypatch):
    s, n = _schedule(what)
    got, launches = _run(s.plan(), [])
    monkeypatch.setenv("POLY_HIP_NO_COPY_DROP", "1")
    want, all_launches = _run(s.plan(), [])
    assert got == want and launches == all_launches - min(n, 1)      # (two copies behind each other are one launch of two kernels)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [11, 33, 300])
@pytest.mark.parametrize("shared", [[], [("logits", "X")], [("W2", "X")], [("b1", "b2")], [("loss", "Y")]])
def test_training_step_on_buffers_that_share_memory(batch, shared, monkeypatch):
    """The logits over the inputs they are made of, a parameter over the batch: the copies of the
    schedule come late, so a step gives the same bits as with each of them launched."""
    s = cases._mlp_schedule(dict(kind="mlp", batch=batch, d_in=50, d_hid=20, d_out=24))
    got, launches = _run(s.plan(), shared)
    monkeypatch.setenv("POLY_HIP_NO_COPY_DROP", "1")
    want, all_launches = _run(s.plan(), shared)
    assert got == want and launches <= all_launches - 5


@pytest.mark.gpu
@pytest.mark.parametrize("shared", [[], [("logits", "X")], [("b1", "b2")]])
def test_profile_leaves_what_a_run_leaves(shared):
    """A timed pass, launch by launch, is a pass: on buffers that share memory, too."""
    import torch
    seen = []
    for timed in (False, True):
        plan = cases._mlp_schedule(dict(kind="mlp", batch=33, d_in=50, d_hid=20, d_out=24)).plan()
        g = torch.Generator(device="cuda")
        g.manual_seed(3)
        data, by = [None] * len(plan.slots), {}
        for slot in plan.external_slots():
            by[slot.name] = data[slot.index] = torch.rand(slot.numel, generator=g, device="cuda")
        for small, large in shared:
            index = [s.index for s in plan.external_slots() if s.name == small][0]
            data[index] = by[small] = by[large][:by[small].numel()]
        for _ in range(2):
            if timed:
                times = plan.profile(data)
                assert len(times) == plan.n_kernels if not shared else len(times) > plan.n_kernels
                assert all(t > 0 for t in times)
            else:
                plan.run(data)
        seen.append({k: v.cpu().numpy().tobytes() for k, v in by.items()})
    assert seen[0] == seen[1]


@pytest.mark.gpu
@pytest.mark.parametrize("what,held,by", [("intermediate", [4], 3), ("copy of a copy", [4, 5], 3), ("update in place", [3], "p")])
def test_where_a_slots_value_is(what, held, by):
    """poly_hip_plan_slot_ptr of a slot whose copy takes no launch: the buffer that holds its value; on buffers
    that share memory, where every kernel is launched, its own again.  The workspace of both forms counts."""
    import ctypes as C

    import torch
    s, _ = _schedule(what)
    plan = s.plan()
    data, index = [None] * len(plan.slots), {}
    for slot in plan.external_slots():
        data[slot.index] = torch.rand(slot.numel, device="cuda")
        index[slot.name] = slot.index

    def value(slot):
        plan.sync()
        host = (C.c_float * N)()
        assert plan.lib.poly_hip_copy_dtoh(host, plan.slot_ptr(slot), 4 * N) == 0
        return list(host)

    plan.run(data)
    at = data[index["p"]].data_ptr() if by == "p" else plan.slot_ptr(by)
    assert at and all(plan.slot_ptr(h) == at for h in held)
    if by == "p":
        small = plan.workspace_bytes()
        data[index["p"]] = data[index["x"]][:N]
        plan.run(data)
        assert plan.slot_ptr(held[0]) not in (None, data[index["p"]].data_ptr()) and value(held[0]) == data[index["p"]].tolist()
        assert plan.workspace_bytes() > small
        data[index["p"]] = torch.rand(N, device="cuda")
        plan.run(data)
        assert plan.slot_ptr(held[0]) == data[index["p"]].data_ptr()
    else:
        want = data[index["x"]].double().reshape(N, K).sum(1)
        assert all(abs(v - w) <= K * 2.0 ** -24 * w for v, w in zip(value(held[0]), want.tolist()))      # (a rounding per term)
