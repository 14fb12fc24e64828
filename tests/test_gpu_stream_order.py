"""A pass of a plan comes after what the caller has queued on torch's current stream --
the default stream or another, busy, idle or never used -- for a plan of one launch, which
is launched directly, and for one that replays a graph."""
import os

import pytest

pytestmark = pytest.mark.gpu

from polygrad_amd import HipPlan
from polygrad_amd.inputs import random_slot_tensors

PLANS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "polygrad_amd", "plans")


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("name,src,out", [("rowops_f32_8192_sum", "a", "sum"), ("mlp_train_f32_b4096", "X", "logits")])
def test_pass_follows_the_callers_stream(name, src, out, own_stream):
    import torch
    plan = HipPlan.from_file(os.path.join(PLANS, name + ".polyplan"))
    frozen = random_slot_tensors(plan, seed=3)
    slot = {s.name: s.index for s in plan.external_slots()}
    x = frozen[slot[src]]
    wanted = {}
    for k in range(3):                       # what a pass gives for the input times k + 1, run on its own
        data = [None if t is None else t.clone() for t in frozen]
        data[slot[src]].mul_(k + 1)
        torch.cuda.synchronize()
        plan.run(data)
        wanted[k] = data[slot[out]].clone()
    assert not torch.equal(wanted[0], wanted[1])
    data = [None if t is None else t.clone() for t in frozen]
    busy = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream() if own_stream else torch.cuda.current_stream()):
        for k in (0, 1, 2, 1, 0):
            for t, f in zip(data, frozen):
                if t is not None:
                    t.copy_(f)
            for _ in range(4 if k else 0):   # (k = 0: the stream is idle again by the time of the pass)
                busy = torch.tanh(busy @ busy)
            data[slot[src]].copy_(x * (k + 1))
            if k == 0:
                torch.cuda.current_stream().synchronize()
            plan.run(data, sync=False)
            plan.sync()
            assert torch.equal(data[slot[out]], wanted[k]), k
    plan.close()
