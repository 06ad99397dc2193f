"""GPU: pgemm_kernel's tiles of 32 and 16 tokens (nl_pgemm.h), at the edges of the rule that chooses them and of the tiles."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_gpu_pgemm import LOGIT_TOL, hip, orc, test_product_against_float64 as _product  # noqa: F401
from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu


# 64-row blocks x 16-token tiles: 1 x 2, 3 x 3, 16 x 16 (256: the last of them), 16 x 17; x 32-token tiles: 32 x 8 (the last), 33 x 9
@pytest.mark.parametrize("rows,cols,n", [(48, 96, 17), (160, 544, 33), (1024, 160, 256), (1008, 288, 257), (2048, 416, 256), (2064, 96, 257)])
@pytest.mark.parametrize("kind", ["q4_0", "q8_0", "f16"])
def test_products(hip, monkeypatch, kind, rows, cols, n):
    _product(hip, monkeypatch, kind, rows, cols, n)


# whole prompts, with the attention's images from 256 tokens on: every epilogue on tiles that share a 64-token group and a 128-key image
@pytest.mark.parametrize("kind,n,bias", [(k, n, n == 289) for k in ("q4_0", "q8_0", "f16") for n in (129, 257, 289, 310)] + [("q4_k", n, False) for n in (17, 47, 130)] + [("q6_k", 33, True)])
def test_prompts_against_the_oracle(hip, orc, tmp_path, kind, n, bias):
    shape = synth.ModelShape("tiles", 2, 384, 6, 2, 512, seq_len=320, interm=640, attn_bias=bias)
    if kind in ("q4_k", "q6_k"):
        shape = synth.ModelShape("tiles", 2, 512, 8, 2, 512, seq_len=320, interm=768, attn_bias=bias)
    p = tmp_path / "t.gguf"
    synth.generate_gguf(str(p), shape, kind, 37)
    g = gguf.load_gguf(str(p))
    toks = synth.prompt_ids(n + 1, shape.vocab, seed=4)
    ref, dev = orc.OracleModel(g), hip.load_llama_model(g)
    orc.set_threads(min(16, os.cpu_count() or 1))
    for pos, tok in enumerate(toks):
        before, want = (want.copy() if pos else None), ref.forward(tok, pos)
    orc.set_threads(1)
    dev.prefill(toks[:n])
    err, bound = float(np.abs(dev.state.logits - before).max()), LOGIT_TOL * max(1.0, float(before.std()))
    assert err <= bound
    dev.forward(toks[n], n)                                  # (reads every row that the prompt stored)
    err, bound = float(np.abs(dev.state.logits - want).max()), LOGIT_TOL * max(1.0, float(want.std()))
    assert err <= bound
    dev.close()
