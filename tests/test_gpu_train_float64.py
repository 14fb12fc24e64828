"""The gradients of one GPT-2 medium block with head and loss, at full size, against the same step in float64
without a rounding on the way: with the vocabulary projection's gradient dealt to workgroups (4096 x 1024 x
100608, parts that a second kernel adds) no further off than summed in one part, whatever the order."""
import math
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

pytestmark = pytest.mark.gpu
B, T, D, H, V = 4, 1024, 1024, 16, 50257
SHAPES = dict(attn_w=(D, 3 * D), proj_w=(D, D), fc_w=(D, 4 * D), fc2_w=(4 * D, D), head_w=(V, D))


def _reference(by):
    import torch
    W = {n: by[n].to(torch.bfloat16).double().reshape(SHAPES.get(n, (-1,))).requires_grad_(True) for n in by if n + ".m" in by}

    def layernorm(x, name):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * W[name + "_w"] + W[name + "_b"]

    h = by["h0"].double().reshape(B, T, D)
    qkv = layernorm(h, "ln1") @ W["attn_w"] + W["attn_b"]
    q, k, v = [t.reshape(B, T, H, D // H).permute(0, 2, 1, 3).reshape(B * H, T, D // H) for t in qkv.split(D, -1)]
    scores = torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(D // H)
    scores = scores.masked_fill(torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1), -1e9)
    ctx = torch.bmm(torch.softmax(scores, -1), v).reshape(B, H, T, D // H).permute(0, 2, 1, 3).reshape(B, T, D)
    h = h + ctx @ W["proj_w"] + W["proj_b"]
    f = layernorm(h, "ln2") @ W["fc_w"] + W["fc_b"]
    f = 0.5 * f * (1 + torch.tanh(0.7978845608028654 * (f + 0.044715 * f ** 3)))
    h = h + f @ W["fc2_w"] + W["fc2_b"]
    loss = torch.nn.functional.cross_entropy(layernorm(h, "lnf").reshape(B * T, D) @ W["head_w"].T, by["target"].long())
    grads = torch.autograd.grad(loss, list(W.values()))
    return loss.detach(), {n: g.reshape(-1) for n, g in zip(W, grads)}


def test_gradients_against_float64(monkeypatch):
    import torch
    want = None
    errors = []
    for one_part in (False, True):
        if one_part:
            monkeypatch.setenv("POLY_HIP_NO_SPLIT_K", "1")
        state = cases.prepare(dict(kind="train"), 21)
        split = [k["desc"] for k in state["plan"].kernel_info() if "K=100608" in k["desc"] and "K dealt to" in k["desc"]]
        assert len(split) == (0 if one_part else 1)
        by = {s.name: state["data"][s.index] for s in state["plan"].external_slots()}
        moments = {n: by[n].double() for n in by if n.endswith(".m")}
        if want is None:
            want = _reference({n: t.clone() for n, t in by.items()})
        cases.run(state)
        state["plan"].sync()
        # the logits are fp32 sums of bf16 products of a bf16 hidden state: an error of each token's loss of
        # some 2^-9 of the logits' spread (0.6), averaged over 4096 tokens
        assert abs(float(by["loss"]) - float(want[0])) <= 4 * 2.0 ** -9 * 0.6 * (B * T) ** -0.5
        # (m = 0.9 m + 0.1 gradient)
        grads = {n: (by[n + ".m"].double() - 0.9 * moments[n + ".m"]) / 0.1 for n in want[1]}
        errors.append({n: float((grads[n] - g).norm() / g.norm()) for n, g in want[1].items()})
        del state, by, moments, grads
        torch.cuda.empty_cache()
    here, one = errors
    for n in want[1]:
        # a few tens of independent roundings to bf16 (2^-9 each) between a weight and its gradient
        if n in SHAPES:
            assert here[n] <= math.sqrt(60) * 2.0 ** -9, (n, here[n])
        # (other roundings of the same kind fall elsewhere: the errors of two orders of summation of one
        # step were seen to differ by up to 2 %, over three sets of inputs)
        assert here[n] <= 1.05 * one[n], (n, here[n], one[n])
