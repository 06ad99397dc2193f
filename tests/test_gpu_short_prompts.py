"""GPU: prompts that end below position 128, and the sampled replies behind them."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nanollama_amd import synth

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUN = """
import sys
import numpy as np
from nanollama_amd import gguf, model, synth
dev = model.load_llama_model(gguf.load_gguf(sys.argv[1]))
out = {}
for n in (8, 40, 127):
    dev.reset()
    dev.prefill(synth.prompt_ids(n, 2048, seed=n))
    assert int(dev.debug_read("step_path", 1)[0]) & 8 == 0
    out[f"logits{n}"] = dev.state.logits.copy()
    u = np.random.default_rng(n).random(24, dtype=np.float32)
    out[f"ids{n}"], _ = dev.sample_decode(n, 24, temperature=0.8, top_p=0.9, top_k=50, rep_penalty=1.15, rep_window=64, uniforms=u, recent=[])
np.savez(sys.argv[2], **out)
dev.close()
"""


@pytest.mark.parametrize("wtype", ["q8_0", "q4_0"])
def test_short_prompts_run_the_tiled_attention(tmp_path, wtype):
    # A sampled reply hangs on the last bits of its prompt (a pick that flips changes all that follow), so a prompt's attention must not depend
    # on where it ends: the kernel that finishes one-split rows of decode batches stays out of it.  NL_NO_ATTN_FIN=1 switches that one off, and makes
    # the tiled kernel leave partials to a merge launch, which are the same bits.
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("short", 4, 576, 9, 3, 2048, seq_len=256, interm=1536), wtype, 71)
    runs = []
    for knob in ({}, {"NL_NO_ATTN_FIN": "1"}):
        to = tmp_path / f"{len(runs)}.npz"
        r = subprocess.run([sys.executable, "-c", RUN, str(p), str(to)], env=dict(os.environ, PYTHONPATH=ROOT, **knob), capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        runs.append(np.load(to))
    for k in runs[0].files:
        assert np.array_equal(runs[0][k], runs[1][k]), k
