"""GPU: prompts of layer-stack models on direct_kernel (nl_mfma.h): every tile its rule chooses, at sizes that fill none of them."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from oracle import stack_oracle as so
from stack_models import BF16_TOL, F32_TOL, config, floats, gla, lat, lconfig, load, rel, tokens, weights

pytestmark = pytest.mark.gpu
TOL = {"float32": F32_TOL, "bfloat16": BF16_TOL}
GATED = lambda width, ff: config([gla(ff=ff)], width=width)
# 64 x 64 (gate and up: 264 row tiles, 19 token tiles); 96 x 128 (33 token tiles, K of 33 tiles); the same for a residual product; 192 x 256 and
# 256 x 256 (500 and 526 row tiles); queries of 40 heads, a row tile of the last one alone
CASES = {"64x64": (GATED(136, 2100), 301), "96x128": (GATED(1032, 2100), 523), "96x128_residual": (GATED(2072, 1032), 1050),
         "192x256": (GATED(72, 4000), 1205), "256x256": (GATED(72, 4200), 1505), "heads": (lconfig([lat(2, heads=41, dim=40, rot=16)]), 301)}


@pytest.mark.parametrize("name,dtype", [(c, "bfloat16") for c in CASES] + [("64x64", "float32"), ("96x128", "float32"), ("heads", "float32")])
def test_long_step_is_the_short_steps(name, dtype):
    cfg, n = CASES[name]
    w, ids, rows = weights(cfg, 93), tokens(n, seed=3), []
    for step in (n, 64):                                   # (64 tokens: few_kernel)
        m = load(cfg, w, dtype, max_streams=1, seq_len=n + 16, max_step_tokens=step)
        rows.append(m.step([(0, ids, 0, [0, n // 2, n - 1])])[0])
        m.close()
    for a, b in zip(*rows):
        assert rel(a, b) < TOL[dtype]                      # (both are within it of the oracle where that is run)


# one tile row and column more or less than a workgroup's
@pytest.mark.parametrize("width,ff,n", [(40, 24, 65), (64, 32, 128), (72, 40, 129), (136, 72, 193)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_edges_against_the_oracle(width, ff, n, dtype):
    cfg = config([gla(ff=ff)], width=width)
    w, ids = weights(cfg, 94), tokens(n, seed=4)
    m = load(cfg, w, dtype, max_streams=1, seq_len=256)
    want = so.forward(cfg, floats(w), ids)
    for a, b in zip(m.step([(0, ids, 0, list(range(n)))])[0], want):
        assert rel(a, b) < TOL[dtype]
    m.close()
