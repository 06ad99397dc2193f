"""GPU: decode batches of layer-stack models with the norm between two products folded around them (MatParams::fw, nl_mfma.h), and the reading
ahead of the next launches' weights (Ahead)."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from oracle import stack_oracle as so
from stack_models import BF16_TOL, F32_TOL, config, floats, gla, load, par, rel, tokens, weights

pytestmark = pytest.mark.gpu


# streams on both sides of a token tile and of what a product's own prologue takes; widths of one and of many k tiles, one (72) that is not
# whole k tiles and keeps its norm launches, one (2080) whose partial sums need a second round; a stream far from magnitude 1; a looped block
@pytest.mark.parametrize("width,n,scale,loop,dtype", [(64, 5, 1.5, None, "float32"), (64, 16, 1.5, (0, 2, 2), "float32"), (96, 17, 1.5, None, "float32"),
                                                      (72, 17, 1.5, None, "float32"), (96, 64, 3e4, None, "float32"), (96, 33, 1e-2, None, "float32"),
                                                      (2080, 3, 1.5, None, "float32"), (2080, 48, 1.5, None, "float32"), (96, 33, 1.5, None, "bfloat16")])
def test_folded_norm_in_decode_batches(width, n, scale, loop, dtype):
    cfg = config([gla(ff=48), par(heads=2, kv=1, ff=32)], width=width, loop=loop, embed_scale=scale)
    w = weights(cfg, 91)
    seqs = [tokens(4 + i % 3, seed=i) for i in range(n)]
    m = load(cfg, w, dtype, max_streams=n, seq_len=32)
    for i, s in enumerate(seqs):
        m.prefill(s[:-2], 0, i, want_logits=False)
    fl = floats(w)
    for back in (2, 1):
        _, rows = m.forward_batch(list(range(n)), [s[-back] for s in seqs], [len(s) - back for s in seqs], want_logits=True)
        for i, s in enumerate(seqs):
            # (the tolerances of the unfolded products: the gains and 1 / rms are applied on the other side of the same sums)
            assert rel(rows[i], so.forward(cfg, fl, s[:len(s) + 1 - back])[-1]) < (F32_TOL if dtype == "float32" else BF16_TOL), (i, back)
    m.close()


# one list, all of them, and a feed-forward past what is read ahead; row tiles and workgroups that are no multiple of the XCDs
@pytest.mark.parametrize("width,ff,n,dtype", [(64, 24, 1, "float32"), (136, 344, 1, "bfloat16"), (136, 344, 40, "float32"), (2056, 2008, 2, "float32")])
def test_weights_read_ahead(monkeypatch, width, ff, n, dtype):
    monkeypatch.setenv("NL_STACK_AHEAD", "1")            # (models of this size otherwise stay in the caches by themselves)
    cfg = config([par(heads=2, kv=1, ff=ff), gla(ff=0), gla(ff=ff)], width=width)
    w = weights(cfg, 92)
    seqs = [tokens(5, seed=50 + i) for i in range(n)]
    m = load(cfg, w, dtype, max_streams=n, seq_len=16)
    for i, s in enumerate(seqs):
        m.prefill(s[:3], 0, i, want_logits=False)
    for at in (3, 4):
        _, rows = m.forward_batch(list(range(n)), [s[at] for s in seqs], [at] * n, want_logits=True)
    fl = floats(w)
    for i, s in enumerate(seqs):
        assert rel(rows[i], so.forward(cfg, fl, s)[-1]) < (F32_TOL if dtype == "float32" else BF16_TOL), i
    m.close()
