"""GPU: the multi-token GEMM of long token runs and of K-quant files (nl_pgemm.h) at the edges of its tiles, tilings and formats."""
import numpy as np
import pytest

from dataclasses import replace

from nanollama_amd import gguf, quant, synth

pytestmark = pytest.mark.gpu

LOGIT_TOL = 1e-4


@pytest.fixture(scope="module")
def hip():
    from nanollama_amd import model
    return model


@pytest.fixture(scope="module")
def orc():
    from oracle import oracle
    return oracle


def _decoded(raw, t, rows, cols):
    if t == gguf.GGML_F16:
        return raw.view(np.float16).astype(np.float64).reshape(rows, cols)
    b = raw.reshape(-1, 34 if t == gguf.GGML_Q8_0 else 18)
    d, q = b[:, :2].copy().view(np.float16).astype(np.float64), b[:, 2:]
    n = q.view(np.int8).astype(np.float64) if t == gguf.GGML_Q8_0 else np.concatenate([(q & 15), (q >> 4)], 1).astype(np.float64) - 8
    return (n * d).reshape(rows, cols)


# tokens and rows that leave ragged tiles, K of whole and of partial 128-column chunks, from a single block on, and 64 x 64 tile counts on every side of the rules:
# <= 256, <= 512, < 1024, above, >= 1792
@pytest.mark.parametrize("rows,cols,n", [(48, 32, 129), (80, 96, 65), (272, 160, 300), (4112, 224, 1801), (16, 512, 65), (80, 544, 127), (272, 576, 129), (1040, 640, 1000), (2064, 512, 1000), (2320, 544, 1801), (4112, 544, 1801)])
@pytest.mark.parametrize("kind", ["q4_0", "q8_0", "f16"])
def test_product_against_float64(hip, monkeypatch, kind, rows, cols, n):
    monkeypatch.setenv("NL_QG2_MIN_TOKENS", "16")            # (small matrices otherwise from the third token tile on)
    t = synth.WTYPES[kind]
    rng = np.random.default_rng(rows + n)
    w, x = rng.standard_normal((rows, cols)).astype(np.float32), rng.standard_normal((n, cols)).astype(np.float32)
    raw = quant.encode(w, t)
    wd, xd = _decoded(raw, t, rows, cols), x.astype(np.float64)
    got = hip.op_matmul_batch(raw, t, x, rows, cols)
    # x = hi + lo leaves 2^-22 of an element, of small ones 2^-25; 32 products and a scaling per block, cols / 32 block sums, each rounded to 2^-24
    bound = (2.0 ** -22 + (cols / 32 + 34) * 2.0 ** -24) * (np.abs(xd) @ np.abs(wd).T) + 2.0 ** -25 * np.abs(wd).sum(1)
    assert (np.abs(got - xd @ wd.T) <= bound).all()


# last groups of one to four pairs, with and without a last odd block, behind whole groups: a group's chunks are its even and its odd blocks, a short one's both
@pytest.mark.parametrize("cols", [288, 320, 352, 384, 416, 448, 480])
@pytest.mark.parametrize("kind", ["q4_0", "q8_0", "f16"])
def test_last_groups_of_a_row(hip, monkeypatch, kind, cols):
    test_product_against_float64(hip, monkeypatch, kind, 272, cols, 129)


class Scaled:
    """A parsed file with the weights of some matrices multiplied by a power of two (their scales, or the fp16 weights themselves)."""

    def __init__(self, g, part, factor):
        self.meta, self.tensor_order, self.g, self.part, self.factor = g.meta, g.tensor_order, g, part, factor

    def get_tensor(self, name):
        raw, info = self.g.get_tensor(name)
        if self.part in name:
            b = np.array(raw).reshape(-1, {gguf.GGML_F16: 2, gguf.GGML_Q8_0: 34, gguf.GGML_Q4_0: 18}[info.type])
            d = (b[:, :2].copy().view(np.float16) * np.float32(self.factor)).astype(np.float16)
            assert np.isfinite(d).all()
            b[:, :2], raw = d.view(np.uint8), b.reshape(-1)
        return raw, info


# a residual stream that grows 2^17-fold in one layer, as far as fp16 scales go: fragments that leave before the norm is known overflow
@pytest.mark.parametrize("kind,n", [("f16", 66), ("f16", 200), ("q8_0", 66), ("q8_0", 300), ("q4_0", 200)])
def test_stream_that_grows_within_a_layer(hip, orc, tmp_path, kind, n):
    shape = replace(synth.TIERS["tiny"], name="grows", dim=576, n_head=9, n_kv_head=3, interm=608, seq_len=320, n_layer=3)
    p = tmp_path / "g.gguf"
    synth.generate_gguf(str(p), shape, kind, 29)
    g = Scaled(gguf.load_gguf(str(p)), "blk.1.ffn_down", 2.0 ** 17)
    toks = synth.prompt_ids(n, shape.vocab, seed=5)
    ref, dev = orc.OracleModel(g), hip.load_llama_model(g)
    for pos, tok in enumerate(toks):
        want = ref.forward(tok, pos)
    dev.prefill(toks)
    assert np.isfinite(want).all() and np.isfinite(dev.state.logits).all()
    assert np.abs(dev.state.logits - want).max() <= LOGIT_TOL * max(1.0, float(want.std()))
    dev.close()


@pytest.mark.parametrize("kind", ["q4_k", "q6_k"])
@pytest.mark.parametrize("n", [3, 16, 64, 65, 200])
def test_kquant_prompt_against_oracle(hip, orc, tmp_path, kind, n):
    # every matrix's epilogue (RoPE + KV store, residual + folded norm, SwiGLU) on super-block weights, in two calls: positions > 0
    shape = replace(synth.TIERS["tiny"], name=f"k_{kind}", dim=512, n_head=8, n_kv_head=2, interm=768, seq_len=256, n_layer=3)
    p = tmp_path / "k.gguf"
    synth.generate_gguf(str(p), shape, kind, 23)
    g = gguf.load_gguf(str(p))
    toks = synth.prompt_ids(n, shape.vocab, seed=3)
    ref, dev = orc.OracleModel(g), hip.load_llama_model(g)
    for pos, tok in enumerate(toks):
        want = ref.forward(tok, pos)
    if n > 100:
        dev.prefill(toks[:37], want_logits=False)
    dev.prefill(toks[37 if n > 100 else 0:], 37 if n > 100 else 0)
    assert np.abs(dev.state.logits - want).max() <= LOGIT_TOL * max(1.0, float(want.std()))
    dev.close()


def test_kquant_streams_equal_the_single_token_plan(hip, tmp_path):
    # decode streams side by side against one forward call each
    shape = replace(synth.TIERS["tiny"], name="k_streams", dim=256, n_head=4, n_kv_head=2, interm=512, seq_len=64)
    p = tmp_path / "s.gguf"
    synth.generate_gguf(str(p), shape, "q4_k", 29)
    g = gguf.load_gguf(str(p))
    dev = hip.load_llama_model(g, max_streams=5)
    for s in range(5):
        for pos in range(s + 1):
            dev.forward(7 + s + pos, pos, s)
    _, rows = dev.forward_batch(list(range(5)), [30, 31, 32, 33, 34], [1, 2, 3, 4, 5], want_logits=True)
    for s in range(5):
        dev.forward(30 + s, s + 1, s)
        assert np.abs(rows[s] - dev.state.logits).max() <= LOGIT_TOL * max(1.0, float(dev.state.logits.std()))
    dev.close()


def test_a_changed_threshold_reaches_recorded_steps(hip, tmp_path, monkeypatch):
    # a decode step's launches are recorded once per geometry: NL_QG2_MIN_TOKENS, read per launch, is part of what they are kept by
    shape = replace(synth.TIERS["tiny"], name="knob", dim=512, n_head=8, n_kv_head=2, interm=768, seq_len=64)
    p = tmp_path / "k.gguf"
    synth.generate_gguf(str(p), shape, "q8_0", 31)
    g = gguf.load_gguf(str(p))

    def step(dev):
        for s in range(8):
            dev.reset(s)
        return dev.forward_batch(list(range(8)), list(range(20, 28)), [0] * 8, want_logits=True)[1].copy()
    dev = hip.load_llama_model(g, max_streams=8)
    split = step(dev)
    monkeypatch.setenv("NL_QG2_MIN_TOKENS", "8")
    changed = step(dev)
    dev.close()
    dev = hip.load_llama_model(g, max_streams=8)
    fresh = step(dev)
    dev.close()
    assert np.array_equal(changed, fresh) and not np.array_equal(changed, split)


# second token tile: matrices of 1536 rows and columns on, smaller ones keep the split-K launches (the same bits as with the other kernel disabled)
@pytest.mark.parametrize("dim,heads,interm,n,moves", [(384, 6, 480, 128, False), (384, 6, 480, 129, True), (576, 9, 1536, 128, False), (576, 9, 1536, 129, True), (1536, 24, 1536, 64, False), (1536, 24, 1536, 65, True)])
@pytest.mark.parametrize("kind", ["q8_0", "f16"])
def test_which_kernel_short_prompts_take(hip, tmp_path, monkeypatch, kind, dim, heads, interm, n, moves):
    shape = replace(synth.TIERS["tiny"], name="route", dim=dim, n_head=heads, n_kv_head=heads // 3, interm=interm, seq_len=192, n_layer=1)
    p = tmp_path / "r.gguf"
    synth.generate_gguf(str(p), shape, kind, 41)
    dev = hip.load_llama_model(gguf.load_gguf(str(p)))
    toks, rows = synth.prompt_ids(n, shape.vocab, seed=9), []
    for knob in (None, "1000000"):
        if knob:
            monkeypatch.setenv("NL_QG2_MIN_TOKENS", knob)
        dev.reset()
        dev.prefill(toks)
        rows.append(dev.state.logits.copy())
    assert np.array_equal(*rows) != moves
    dev.close()
