"""GPU: pgemm_kernel's tiles of 16 rows for short prompts of Q6_K files (nl_pgemm.h): the bits of the 64-row tiles, over odd numbers of
row tiles, last groups of one to three pairs, every edge of the token tiles, biases, and matrices on both sides of the rule."""
import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu

# layers, width, query heads, kv heads, feed-forward, options
SHAPES = {
    "odd": (2, 768, 12, 3, 1280, {}),                                # 72, 48 and 80 row tiles, six to ten 128-column chunks
    "narrow": (2, 256, 4, 2, 768, {}),
    "heads32": (2, 512, 16, 4, 512, {}),
    "bias": (2, 512, 8, 1, 1024, dict(attn_bias=True)),
    "wide_ff": (1, 256, 4, 1, 8448, {}),                              # gate and up together 264 blocks of 64 rows: the rule says no
}


@pytest.mark.parametrize("wtype", ["q6_k", "q4_k"])
@pytest.mark.parametrize("name", SHAPES)
def test_the_bits_of_the_larger_tiles(tmp_path, monkeypatch, name, wtype):
    from nanollama_amd import model
    layers, dim, heads, kvs, ff, opts = SHAPES[name]
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape(name, layers, dim, heads, kvs, 256, seq_len=160, interm=ff, **opts), wtype, 41)
    m = model.load_llama_model(gguf.load_gguf(str(p)))
    toks = [int(t) for t in np.random.default_rng(3).integers(3, 256, size=160)]
    for n, at in ((8, 0), (16, 0), (17, 0), (33, 0), (63, 0), (64, 0), (65, 0), (48, 100), (30, 11)):
        rows, path = [], []
        for knob in ("1", "0"):
            monkeypatch.setenv("NL_PG_SLIM", knob)
            m.reset()
            if at:
                m.prefill(toks[:at], 0, want_logits=False)
            m.prefill(toks[at:at + n], at)
            path.append(int(m.debug_read("step_path", 1)[0]) & 256)
            rows.append(m.state.logits.copy())
            m.forward(toks[0], at + n)                              # (reads every row that the prompt stored)
            rows.append(m.state.logits.copy())
        assert path == [256 if n <= 64 and name != "wide_ff" and wtype == "q6_k" else 0, 0], n
        assert np.isfinite(rows[0]).all() and np.array_equal(rows[0], rows[2]) and np.array_equal(rows[1], rows[3]), (n, at, float(np.abs(rows[0] - rows[2]).max()))
    m.close()
