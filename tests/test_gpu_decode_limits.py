"""GPU: which decode launch serves which position on wide tiers (one GPU), and that both sides of every limit agree."""
import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu


# Q4_0: a head's passes are shared with three blocks of its own kv group (positions 256 .. 1023); Q8_0: one runner, the first pass only
@pytest.mark.parametrize("wtype,limit", [("q4_0", 1024), ("q8_0", 256)])
def test_fused_launch_against_the_general_plan_at_every_pass(tmp_path, monkeypatch, wtype, limit):
    from nanollama_amd import model as hip
    shape = synth.ModelShape("limits", 2, 1536, 24, 6, 512, seq_len=1100, interm=2048)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, wtype, 83, mode="qrand")
    g = gguf.load_gguf(str(p))
    dev = hip.load_llama_model(g)
    info = dev.plan_info()
    assert info["fused_mode"] == 4 and info["fused_max_pos"] == limit, info
    monkeypatch.setenv("NL_FUSED_ATTN", "0")
    plain = hip.load_llama_model(g)
    toks = synth.prompt_ids(1050, shape.vocab, seed=11)
    for m in (dev, plain):
        m.prefill(toks, want_logits=False)
    for pos in (0, 15, 16, 254, 255, 256, 257, 511, 512, 700, 767, 768, 1022, 1023, 1024, 1040):
        for m in (dev, plain):
            m.forward(toks[pos] % 500 + 3, pos)
        # (float32 sums in another order through two layers)
        assert np.abs(dev.state.logits - plain.state.logits).max() <= 1e-4 * max(1.0, float(plain.state.logits.std())), pos
    assert dev.decode_greedy(5, 250, 12) == plain.decode_greedy(5, 250, 12)        # across the first pass's end
    assert dev.decode_greedy(5, 1018, 12) == plain.decode_greedy(5, 1018, 12)      # and across the limit of the shared ones
    assert dev.last_error() == ""
    dev.close(); plain.close()


def test_two_passes_per_helper_of_the_kv_group(tmp_path, monkeypatch):
    # 24 kv groups of 2 heads and 192 output tiles: no blocks past the groups, the feed-forward half in one launch -- a head's passes 0 .. 6 are
    # shared with three blocks of its own group, two each from position 1024 on
    from nanollama_amd import model as hip
    shape = synth.ModelShape("limits_wide", 2, 3072, 48, 24, 512, seq_len=2048, interm=3072)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, "q4_0", 84, mode="qrand")
    g = gguf.load_gguf(str(p))
    dev = hip.load_llama_model(g)
    info = dev.plan_info()
    assert info["fused_mode"] == 4 and info["fused_max_pos"] == 2048, info
    monkeypatch.setenv("NL_FUSED_ATTN", "0")
    plain = hip.load_llama_model(g)
    toks = synth.prompt_ids(2040, shape.vocab, seed=12)
    for m in (dev, plain):
        m.prefill(toks, want_logits=False)
    for pos in (255, 256, 1023, 1024, 1279, 1280, 1535, 1536, 1792, 2046):
        for m in (dev, plain):
            m.forward(toks[min(pos, 2039)] % 500 + 3, pos)
        assert np.abs(dev.state.logits - plain.state.logits).max() <= 1e-4 * max(1.0, float(plain.state.logits.std())), pos
    assert dev.decode_greedy(5, 1018, 12) == plain.decode_greedy(5, 1018, 12)
    assert dev.last_error() == ""
    dev.close(); plain.close()
