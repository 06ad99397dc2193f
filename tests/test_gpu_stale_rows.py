"""GPU: cache rows that an earlier conversation left are nobody's operands, not even times zero: Reset (go/model.go:623-631) drops them, and a row that is not
finite must not reach the next conversation through the masked positions of a pass.  Every launch plan of a single token, and the prompt's."""
import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu

# plan: weights, layers, width, query heads, kv heads, feed-forward, vocabulary, knobs
PLANS = {
    "layers": ("q8_0", 2, 768, 12, 3, 1280, 512, dict(NL_LAYERS="2")),
    "layers_k": ("q4_k", 2, 1024, 16, 2, 2048, 512, dict(NL_LAYERS="2")),
    "blocks": ("q4_0", 3, 768, 12, 3, 2048, 512, dict(NL_LAYERS="0")),
    "projection": ("q8_0", 2, 1024, 16, 4, 1024, 512, dict(NL_LAYERS="0", NL_FUSED_ATTN="2")),
    "wide": ("q4_0", 2, 1536, 24, 6, 4096, 512, dict(NL_LAYERS="0")),
    "general": ("q8_0", 2, 768, 12, 3, 1280, 512, dict(NL_LAYERS="0", NL_FUSED_ATTN="0")),
    "persistent": ("q8_0", 13, 576, 9, 9, 1536, 32000, dict()),
}
MODE = {"layers": None, "layers_k": 0, "blocks": 1, "projection": 2, "wide": 4, "general": 0, "persistent": 1}


@pytest.mark.parametrize("plan", PLANS)
def test_rows_of_an_earlier_conversation(tmp_path, monkeypatch, plan):
    from nanollama_amd import model as hip
    wtype, layers, dim, heads, kv, ff, vocab, knobs = PLANS[plan]
    for k, v in knobs.items():
        monkeypatch.setenv(k, v)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape(plan, layers, dim, heads, kv, vocab, seq_len=320, interm=ff), wtype, 21, mode="qrand")
    g = gguf.load_gguf(str(p))
    dev, clean = hip.load_llama_model(g), hip.load_llama_model(g)
    assert MODE[plan] is None or dev.plan_info()["fused_mode"] == MODE[plan]
    assert dev.persist_info()["ready"] == (plan == "persistent")
    dev.set_gamma(np.array([7], np.int32), np.full((1, dim), np.nan, np.float32))
    toks = synth.prompt_ids(300, vocab, seed=2)
    for pos in (0, 1, 15, 16, 40, 127, 128, 200):
        dev.reset()
        dev.set_gamma(np.array([7], np.int32), np.full((1, dim), np.nan, np.float32))
        dev.prefill([7] * 300)
        assert not np.isfinite(dev.state.logits).any()
        dev.set_gamma(np.zeros(0, np.int32), np.zeros((0, dim), np.float32))
        dev.reset()
        clean.reset()
        for m in (dev, clean):
            if pos:
                m.prefill(toks[:pos], want_logits=False)
            m.forward(toks[pos], pos)
        assert np.isfinite(clean.state.logits).all() and np.array_equal(dev.state.logits, clean.state.logits), pos
        assert dev.decode_greedy(toks[pos + 1], pos + 1, 20) == clean.decode_greedy(toks[pos + 1], pos + 1, 20), pos
    dev.close(); clean.close()
