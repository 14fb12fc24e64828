"""The on-device search (POLY_BEAM) over products of few or ragged tiles, fp32 ones on bf16 planes and attention of few,
ragged or fp32 queries and keys: they bring candidates, each of which runs, and what the
search decides changes no bit."""
import os
import re

import pytest

from test_small_matmul import _case, cases

pytestmark = pytest.mark.gpu

# case, kernels that have candidates: what their descriptions say, and the label of one
CASES = [(_case(100, 300, 515, "bfloat16", "nn"), "depth dealt to", "32x32w8x6p1"), (_case(12, 770, 1000, "float16", "tn"), "depth dealt to", "16x16w8x6p1"),
         (_case(128, 768, 768, "float32", "nt"), "depth dealt to", "f32_32x32w4x6"), (_case(345, 776, 2304, "float32", "nn"), "of two sums each", "f32_64x64w4x4"),
         (_case(1111, 999, 601, "bfloat16", "nn"), "rows of any alignment", "128x128x64w2x4s2g1"), (_case(1500, 1401, 130, "float16", "tn"), "rows of any alignment", "64x64x64w2x2s2g2"),
         (_case(1030, 1040, 97, "float32", "nn"), "three planes", "f32_64x64w2x2"), (_case(1801, 1700, 160, "float32", "tn"), "three planes", "f32_128x128w4x2"),
         (cases._gpt2(3, 40, "bfloat16", layers=1), "scores of", "attn_occ2"), (cases._gpt2(1, 130, "float32", layers=1), "scores of", "attn_occ4")]


@pytest.mark.parametrize("case,what,label", CASES, ids=lambda v: v if isinstance(v, str) else v["kind"])
def test_search_has_candidates_and_changes_no_bit(case, what, label, tmp_path, monkeypatch, capfd):
    import torch
    monkeypatch.setenv("POLY_HIP_CACHE_DIR", str(tmp_path))

    def outputs():
        state = cases.prepare(case, 3)
        for t in state["out"].values():
            t.fill_(float("nan"))
        for _ in range(2):
            cases.run(state)
        state["plan"].sync()
        desc = [k["desc"] for k in state["plan"].kernel_info()]
        out = [t.clone() for t in state["out"].values()]
        state["plan"].close()
        return out, desc

    want, desc = outputs()
    assert any(what in d for d in desc), desc
    monkeypatch.setenv("POLY_BEAM", "1")
    monkeypatch.setenv("POLY_HIP_DEBUG", "1")
    capfd.readouterr()
    got, _ = outputs()
    lines = [ln for ln in capfd.readouterr().err.splitlines() if ln.startswith("polygrad: tune: ") and what in ln]
    timed = dict(re.findall(r" (\S+)=(-?[0-9.]+)", lines[0][lines[0].index("(ms:"):].rstrip(")")))
    assert {"default", label} <= set(timed) and all(float(t) > 0 for t in timed.values()), lines[0]
    assert all(torch.isfinite(t.float()).all() for t in want) and all(torch.equal(a, b) for a, b in zip(want, got))
    assert any(f.endswith(".tune") for f in os.listdir(tmp_path))
