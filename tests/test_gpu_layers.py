"""GPU: all layers of a decode step in one launch (nl_layers.h) against the five-launch plan, at the edges of its passes, units and column groups."""
import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu

# layers, width, query heads, kv heads, feed-forward, options; positions
SHAPES = {
    "middle": ((2, 1536, 24, 6, 4096, {}), (0, 1, 15, 16, 126, 127, 128, 129, 255, 256, 640, 1030)),                    # the largest feed-forward: a tile a workgroup
    "ragged": ((3, 576, 9, 9, 1472, {}), (0, 17, 127, 128, 300)),                                                      # last groups of one and three pairs
    "small": ((2, 128, 2, 1, 192, {}), (0, 5, 127, 128, 140)),                                                         # half a group a row
    "widest": ((2, 2048, 32, 8, 4096, {}), (0, 127, 128, 1023, 1024, 1100, 2046)),                                     # from 1024 on two heads a unit
    "wide_groups": ((2, 768, 12, 3, 1280, {}), (0, 31, 127, 128, 260)),                                                # 256-column groups, the last shares of five
    "eight_to_one": ((2, 1024, 16, 2, 2048, {}), (3, 200, 2040)),
    "variant": ((2, 768, 12, 3, 2048, dict(rope_conjugate=True, attn_bias=True)), (0, 60, 127, 128, 200)),
}


def _models(tmp_path, monkeypatch, name, wtype, vocab=512, seq_len=2048):
    from nanollama_amd import model as hip
    (layers, dim, heads, kv, ff, opts), _ = SHAPES[name]
    shape = synth.ModelShape(name, layers, dim, heads, kv, vocab, seq_len=seq_len, interm=ff, **opts)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, wtype, 91, mode="qrand")
    g = gguf.load_gguf(str(p))
    monkeypatch.setenv("NL_LAYERS", "2")
    dev = hip.load_llama_model(g)
    monkeypatch.setenv("NL_LAYERS", "0")
    monkeypatch.setenv("NL_FUSED_ATTN", "0")
    plain = hip.load_llama_model(g)
    return shape, dev, plain


@pytest.mark.parametrize("name,wtype", [(n, w) for n in SHAPES for w in ("q8_0", "q4_0")] + [("middle", "q5_0")] +
                         [(n, w) for n in ("middle", "wide_groups", "eight_to_one") for w in ("q4_k", "q6_k")])
def test_against_the_five_launch_plan(tmp_path, monkeypatch, name, wtype):
    shape, dev, plain = _models(tmp_path, monkeypatch, name, wtype)
    assert dev.debug_read("layers_max_pos", 1)[0] == 2048 and plain.debug_read("layers_max_pos", 1)[0] == 0
    positions = SHAPES[name][1]
    toks = synth.prompt_ids(max(positions) + 1, shape.vocab, seed=11)
    for m in (dev, plain):
        m.prefill(toks, want_logits=False)
    for pos in positions:
        for m in (dev, plain):
            m.forward(toks[pos] % 500 + 3, pos)
        # (float32 sums in another order through two or three layers)
        assert np.abs(dev.state.logits - plain.state.logits).max() <= 1e-4 * max(1.0, float(plain.state.logits.std())), pos
    n = shape.n_layer * shape.n_kv_head * shape.seq_len * 64
    for which in ("k_cache", "v_cache"):       # rows that both wrote at those positions, of values up to 10
        a, b = dev.debug_read(which, n).reshape(-1, shape.seq_len, 64), plain.debug_read(which, n).reshape(-1, shape.seq_len, 64)
        assert np.abs(a - b).max() <= 1e-4
    assert dev.decode_greedy(5, 120, 40) == plain.decode_greedy(5, 120, 40)        # graphs of sixteen steps and single ones, across a pass
    assert dev.last_error() == ""
    dev.close(); plain.close()


def test_streams_and_sampled_chains(tmp_path, monkeypatch):
    from nanollama_amd import model as hip
    (layers, dim, heads, kv, ff, opts), _ = SHAPES["middle"]
    shape = synth.ModelShape("streams", layers, dim, heads, kv, 512, seq_len=300, interm=ff)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, "q8_0", 92, mode="qrand")
    g = gguf.load_gguf(str(p))
    out = []
    for knob in ("2", "0"):
        monkeypatch.setenv("NL_LAYERS", knob)
        m = hip.load_llama_model(g, max_streams=3)
        assert (m.debug_read("layers_max_pos", 1)[0] > 0) == (knob == "2")
        got = []
        for s, n in ((2, 140), (0, 20)):
            toks = synth.prompt_ids(n, shape.vocab, seed=s)
            m.prefill(toks, 0, s)
            ids, _ = m.sample_decode(n, 37, temperature=0.8, top_p=0.9, top_k=50, rep_penalty=1.15, rep_window=64,
                                     uniforms=np.random.default_rng(s).random(37, dtype=np.float32), recent=[], stream=s)
            got.append(ids)
        out.append(got)
        m.close()
    assert out[0] == out[1]


def test_a_wait_that_gives_up_is_redone_on_the_five_launch_plan(tmp_path, monkeypatch):
    monkeypatch.setenv("NL_FUSED_SPIN_LIMIT", "0")
    monkeypatch.setenv("NL_QUIET", "1")
    shape, dev, plain = _models(tmp_path, monkeypatch, "variant", "q8_0")
    toks = synth.prompt_ids(6, shape.vocab, seed=3)
    for pos, t in enumerate(toks):
        for m in (dev, plain):
            m.forward(t, pos)
        assert np.array_equal(dev.state.logits, plain.state.logits), pos
    assert "timed out" in dev.last_error() and dev.debug_read("layers_max_pos", 1)[0] == 0
    dev.close(); plain.close()


@pytest.mark.parametrize("layers,wtype,runs", [(2, "q8_0", False), (4, "q8_0", True), (4, "q4_k", True), (4, "f16", False)])
def test_models_that_take_the_launch(tmp_path, monkeypatch, layers, wtype, runs):
    from nanollama_amd import model as hip
    monkeypatch.delenv("NL_LAYERS", raising=False)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("rule", layers, 1024, 16, 4, 512, seq_len=160, interm=1024), wtype, 5, mode="qrand")
    m = hip.load_llama_model(gguf.load_gguf(str(p)))
    assert m.debug_read("layers_max_pos", 1)[0] == (160 if runs else 0)
    m.close()


# forwards since the launch last wrote its buffers (here: since they were cleared): half the counter's range back is not ahead
@pytest.mark.parametrize("counter", [0x7ffff0, 0x7fffff, 0x800000, 0xfffff0, 0xffffff, 0x1000000])
def test_the_age_of_a_buffer_does_not_matter(tmp_path, monkeypatch, counter):
    monkeypatch.setenv("NL_FORWARD_COUNTER", str(counter))
    monkeypatch.setenv("NL_QUIET", "1")
    shape, dev, plain = _models(tmp_path, monkeypatch, "wide_groups", "q8_0", seq_len=300)
    toks = synth.prompt_ids(20, shape.vocab, seed=3)
    for m in (dev, plain):
        m.prefill(toks, want_logits=False)
    assert dev.decode_greedy(5, 20, 40) == plain.decode_greedy(5, 20, 40)
    assert dev.last_error() == "" and dev.debug_read("layers_max_pos", 1)[0] > 0
    dev.close(); plain.close()


# a launch that gives up (it met another process's on the card, say) is tried again; the plans that served its positions before outlive it
@pytest.mark.parametrize("name,wtype,mode", [("middle", "q4_k", 0), ("variant", "q8_0", 1), ("middle", "q8_0", 4)])
def test_three_give_ups(tmp_path, monkeypatch, name, wtype, mode):
    monkeypatch.setenv("NL_FUSED_SPIN_LIMIT", "0")
    monkeypatch.setenv("NL_QUIET", "1")
    shape, dev, plain = _models(tmp_path, monkeypatch, name, wtype, seq_len=300)
    toks = synth.prompt_ids(30, shape.vocab, seed=3)
    for m in (dev, plain):
        m.prefill(toks, want_logits=False)
        m.reset()
    state = lambda: (dev.debug_read("layers_max_pos", 1)[0], dev.plan_info()["fused_mode"])
    assert state() == (300, mode) and dev.last_error() == ""
    for m in (dev, plain):
        m.forward(toks[0], 0)
    assert np.array_equal(dev.state.logits, plain.state.logits)
    assert state() == (300, mode) and "timed out" in dev.last_error() and "tries" in dev.last_error()
    assert dev.decode_greedy(toks[1], 1, 37) == plain.decode_greedy(toks[1], 1, 37)
    assert state() == (300, mode)
    us = np.random.default_rng(9).random(20, dtype=np.float32)
    assert dev.sample_decode(38, 20, 0.9, 0.9, 50, 1.15, 8, us, [3, 4]) == plain.sample_decode(38, 20, 0.9, 0.9, 50, 1.15, 8, us, [3, 4])
    assert state() == (0, mode)                                 # ... the third
    for m in (dev, plain):
        m.forward(toks[5], 58)
    assert np.array_equal(dev.state.logits, plain.state.logits)
    assert state() == (0, 0)                                    # (a fused plan gave up as well, once)
    dev.close(); plain.close()


# a replay without a forward of its own finds every granule already there, and what it times leaves the exchanges out
def test_profiled_replays_are_forwards(tmp_path, monkeypatch):
    shape, dev, plain = _models(tmp_path, monkeypatch, "middle", "q8_0", seq_len=300)
    assert dev.layers_info() == {"min_pos": 0, "max_pos": 300, "launches": 4} and plain.layers_info() == {"min_pos": 0, "max_pos": 0, "launches": 0}
    toks = synth.prompt_ids(20, shape.vocab, seed=3)
    for m in (dev, plain):
        m.prefill(toks, want_logits=False)
    before = dev.debug_read("forwards", 1)[0]
    kinds = {k: c for k, (ms, c) in dev.profile_forward(5, 20, iters=7).items() if c}
    assert kinds == {"embed": 1, "ffn_block": 1, "lm_head": 1, "argmax": 1}
    assert dev.debug_read("forwards", 1)[0] - before == 1 + 7 + 7           # one ahead, the embed launch's replays, the layer launch's
    assert dev.last_error() == ""
    for m in (dev, plain):
        m.forward(5, 20)
    assert np.abs(dev.state.logits - plain.state.logits).max() <= 1e-4 * max(1.0, float(plain.state.logits.std()))
    dev.close(); plain.close()


@pytest.mark.parametrize("layers,dim,heads,min_pos", [(4, 256, 4, 384), (7, 256, 4, 384), (8, 256, 4, 256), (4, 1024, 16, 0)])
def test_where_the_launch_takes_over(tmp_path, monkeypatch, layers, dim, heads, min_pos):
    from nanollama_amd import model as hip
    monkeypatch.delenv("NL_LAYERS", raising=False)
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("rule", layers, dim, heads, 2, 512, seq_len=512, interm=1024), "q8_0", 5, mode="qrand")
    m = hip.load_llama_model(gguf.load_gguf(str(p)))
    assert m.layers_info()["min_pos"] == min_pos and m.layers_info()["max_pos"] == 512
    m.close()


def _plan(m):
    return int(m.debug_read("plan", 1)[0])


# two launches a layer below position 256, one launch for all from there on: what ran on both sides, and a greedy chain across against the handle that keeps the former
def test_the_launch_takes_over_within_a_chain(tmp_path, monkeypatch):
    from nanollama_amd import model as hip
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("over", 8, 768, 12, 3, 512, seq_len=400, interm=2048), "q8_0", 97, mode="qrand")
    g = gguf.load_gguf(str(p))
    monkeypatch.delenv("NL_LAYERS", raising=False)
    dev = hip.load_llama_model(g)
    monkeypatch.setenv("NL_LAYERS", "0")
    blocks = hip.load_llama_model(g)
    assert dev.layers_info()["min_pos"] == 256 and blocks.plan_info()["fused_mode"] == 1
    toks = synth.prompt_ids(400, 512, seed=4)
    for m in (dev, blocks):
        m.prefill(toks[:254], want_logits=False)
    for pos, plan in ((254, 1), (255, 1), (256, 3), (257, 3)):
        for m in (dev, blocks):
            m.forward(toks[pos], pos)
        assert (_plan(dev), _plan(blocks)) == (plan, 1), pos
        assert np.abs(dev.state.logits - blocks.state.logits).max() <= 1e-4 * max(1.0, float(blocks.state.logits.std())), pos
    ids = [m.decode_greedy(7, 200, 150) for m in (dev, blocks)]
    assert ids[0] == ids[1] and (_plan(dev), _plan(blocks)) == (3, 1)
    dev.close(); blocks.close()


# more positions than units for them: 20 kv heads have 12 of 128 positions each, and the launch ends there
def test_the_launch_ends_below_the_context(tmp_path, monkeypatch):
    from nanollama_amd import model as hip
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("ends", 2, 1280, 20, 20, 512, seq_len=2048, interm=1024), "q8_0", 98, mode="qrand")
    g = gguf.load_gguf(str(p))
    monkeypatch.setenv("NL_LAYERS", "2")
    monkeypatch.setenv("NL_FUSED_MAX_POS", "0")
    dev = hip.load_llama_model(g)
    monkeypatch.setenv("NL_LAYERS", "0")
    monkeypatch.setenv("NL_FUSED_ATTN", "0")
    plain = hip.load_llama_model(g)
    assert dev.layers_info()["max_pos"] == 1536
    toks = synth.prompt_ids(2048, 512, seed=4)
    for m in (dev, plain):
        m.prefill(toks[:1534], want_logits=False)
    for pos, plan in ((1534, 3), (1535, 3), (1536, 0), (1537, 0)):
        for m in (dev, plain):
            m.forward(toks[pos], pos)
        assert _plan(dev) == plan, pos
        assert np.abs(dev.state.logits - plain.state.logits).max() <= 1e-4 * max(1.0, float(plain.state.logits.std())), pos
    assert dev.decode_greedy(7, 1500, 60) == plain.decode_greedy(7, 1500, 60)
    assert dev.last_error() == ""
    dev.close(); plain.close()


@pytest.mark.parametrize("name,wtype", [("middle", "q8_0"), ("wide_groups", "q4_0"), ("eight_to_one", "q4_k"), ("middle", "q6_k")])
def test_every_call_runs_on_the_launch(tmp_path, monkeypatch, name, wtype):
    shape, dev, plain = _models(tmp_path, monkeypatch, name, wtype, seq_len=300)
    for m, plan in ((dev, 3), (plain, 0)):
        m.prefill([5, 6])
        assert _plan(m) == plan
        m.forward(7, 2)
        assert _plan(m) == plan
        m.forward_argmax(8, 3)
        assert _plan(m) == plan
        m.decode_greedy(9, 4, 20)
        assert _plan(m) == plan
        m.sample_decode(24, 20, 0.9, 0.9, 50, 1.15, 8, np.linspace(0, 0.99, 20, dtype=np.float32), [3, 4])
        assert _plan(m) == plan
        m.forward_batch([0], [7], [44])
        assert _plan(m) == plan
    dev.close(); plain.close()
