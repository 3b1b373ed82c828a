"""Which runs bench.py compares token by token: those that were fed the same tokens."""
import importlib

import pytest


@pytest.mark.parametrize("prompt,warmup,compared", [(440, 8, True), (487, 5, False), (400, 8, False)])
def test_graph_case_is_compared_with_a_headline_behind_the_same_prompt(lva, monkeypatch, prompt, warmup, compared):
    bench, measure = importlib.import_module("bench"), importlib.import_module("llama-vulkan_amd.measure")
    expected = {}

    def decode_case(ctx, name, *args, expect_picks=None, **kw):
        expected[name] = expect_picks
        return dict(path="graph", tok_s=1.0, ms_per_token=1.0, GBps=1.0, frac_of_peak=1.0, picks=[5, 6])
    monkeypatch.setattr(measure, "decode_case", decode_case)
    monkeypatch.setattr(measure, "gemv_cases", lambda *a, **k: [])
    monkeypatch.setattr(measure, "gemm_cases", lambda *a, **k: [])
    monkeypatch.setattr(measure, "prefill_case", lambda *a, **k: dict(tok_s=1.0, ms=1.0, TFLOPs=1.0, executed_TFLOPs=1.0, frac_of_mfma_peak=1.0, executed_frac=1.0))
    picks = [7, 8, 9]
    cases = bench.other_cases(lva, None, headline_picks=picks, headline_first=prompt + warmup, headline_prompt=prompt)
    row = [c for c in cases if c["name"].startswith("7B q4_0 decode, positions 444")][0]
    assert row["same_tokens_as"] == ("headline" if compared else None)
    assert expected["decode-13b-graph"] == [5, 6]
    want = expected["decode-7b-graph"]
    if compared:
        assert want[warmup:] == picks and len(want) == warmup + 3 and all(w == 1 for w in want[:warmup])
    else:
        assert want is None
