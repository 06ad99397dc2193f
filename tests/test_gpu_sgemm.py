"""GPU tests of the short multi-token steps on sgemm_kernel (nanollama_amd/csrc/nl_sgemm.h): Q8_0, F16 and Q4_0 files, any width of whole
32-value blocks.  The kernel takes qgemm_kernel's K splits in qgemm_kernel's order, so the same handle's split-K launches (NL_SGEMM=0) give the
same bits here: rows, logits and cache (its norm agrees with bnorm_kernel's to a few float64 ulps, which a float32 factor all but never shows).  Reference: go/model.go:510-612 per stream, go/quant.go:45-165, :527-563."""
import os
import sys

import numpy as np
import pytest

from nanollama_amd import gguf, synth

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu

SHAPES = {
    # three blocks and seven: a last chunk, group and pair that are not whole; head_dim 32, grouped heads, biases
    "d96_i224": synth.ModelShape("sg_a", 2, 96, 3, 1, 160, seq_len=160, interm=224, attn_bias=True),
    # the smallest tier's widths (two and a quarter groups), conjugate rotation
    "d576_i1536": synth.ModelShape("sg_b", 2, 576, 9, 3, 256, seq_len=160, interm=1536, rope_conjugate=True),
    # few rows, long columns: sixteen splits of the down projection; a group of three pairs
    "d160_i4000": synth.ModelShape("sg_c", 1, 160, 5, 5, 96, seq_len=96, interm=4000),
    # two row tiles a wavefront from 33 tokens on, six chunks a split
    "d1536_i4096": synth.ModelShape("sg_d", 1, 1536, 24, 6, 128, seq_len=96, interm=4096),
    # eight blocks a wavefront; sixteen wavefronts with a fifth block for two of them, the widest token tile that LDS holds; the first one that it does not
    "d2048_i5632": synth.ModelShape("sg_e", 1, 2048, 32, 8, 128, seq_len=96, interm=5632),
    "d2112_i704": synth.ModelShape("sg_f", 1, 2112, 33, 11, 128, seq_len=96, interm=704),
    "d2144_i704": synth.ModelShape("sg_g", 1, 2144, 67, 67, 128, seq_len=96, interm=704),
}


def short_step(m):
    """Did the last multi-token step run on sgemm_kernel?"""
    return int(m.debug_read("step_path", 1)[0]) & 2 != 0


@pytest.fixture(scope="module")
def hip():
    from nanollama_amd import _lib, model
    if _lib.lib().nl_device_count() < 1:
        pytest.fail("no HIP device visible: the GPU tests must run on the MI355X box")
    return model


@pytest.mark.parametrize("wtype", ["q8_0", "f16", "q4_0", "q5_0"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_short_steps_give_the_bits_of_the_split_k_launches(hip, tmp_path, monkeypatch, name, wtype):
    monkeypatch.setenv("NL_DGEMM", "0")                  # (widths of whole 256-column groups too)
    shape = SHAPES[name]
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, wtype, 17)
    m = hip.load_llama_model(gguf.load_gguf(str(p)), max_streams=40)
    rng = np.random.default_rng(3)
    toks = [int(t) for t in rng.integers(3, shape.vocab, size=shape.seq_len)]
    for n in (3, 9, 16, 17, 48, 64, 70):
        got = {}
        for knob in ("0", "2"):                          # (2: wherever the kernel can, however many rounds of workgroups it takes)
            monkeypatch.setenv("NL_SGEMM", knob)
            m.reset()
            m.prefill(toks[:n])
            # beyond 64 tokens the wide shapes' unsplit products are more than six chunks long
            assert short_step(m) == (knob == "2" and shape.dim <= 2112 and (n <= 64 or shape.dim < 1536)), (n, knob)
            rows = [m.state.logits.copy()]
            m.prefill(toks[n:n + 9], n)                  # over the rows that the first prompt left in the cache
            got[knob] = rows + [m.state.logits.copy()]
        for a, b in zip(got["0"], got["2"]):
            assert np.isfinite(a).all() and np.array_equal(a, b), (n, float(np.abs(a - b).max()))
    for ns, ctx in ((3, 5), (40, 5), (21, 80)):
        ctx = min(ctx, shape.seq_len - 4)
        got = {}
        for knob in ("0", "2"):
            monkeypatch.setenv("NL_SGEMM", "0")
            for s in range(ns):
                m.reset(s)
                m.prefill(toks[s % 7:][:ctx - s % 3], 0, s, want_logits=False)
            monkeypatch.setenv("NL_SGEMM", knob)
            got[knob] = [m.forward_batch(list(range(ns)), toks[i:i + ns], [ctx - s % 3 + i for s in range(ns)], want_logits=True)[1].copy() for i in range(3)]
            assert short_step(m) == (knob == "2" and shape.dim <= 2112), (ns, ctx, knob)
        for a, b in zip(got["0"], got["2"]):
            assert np.isfinite(a).all() and np.array_equal(a, b), (ns, ctx, float(np.abs(a - b).max()))
    m.close()


@pytest.mark.parametrize("wtype", ["q8_0", "f16"])
def test_short_steps_match_the_oracle(hip, tmp_path, wtype):
    from oracle import oracle
    shape = SHAPES["d576_i1536"]
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, wtype, 18)
    g = gguf.load_gguf(str(p))
    toks = [int(t) for t in np.random.default_rng(4).integers(3, shape.vocab, size=29)]
    ref = oracle.OracleModel(g)
    for pos, t in enumerate(toks):
        want = ref.forward(t, pos)
    m = hip.load_llama_model(g)
    m.prefill(toks)
    assert short_step(m)
    assert float(np.abs(m.state.logits - want).max()) <= 1e-4 * max(1.0, float(want.std()))
    m.close()


# steps of four to eight rounds of workgroups, either side of the limits: sgemm_kernel up to the last of them
@pytest.mark.parametrize("dim,heads,kvs,interm,wtype,stream_steps,prompts", [
    (1600, 25, 25, 4288, "q8_0", {17: True, 48: True, 49: False, 64: False}, {48: True, 49: False}),
    (1600, 25, 25, 4288, "q4_0", {48: True, 49: False}, {49: True, 64: True}),
    (2112, 33, 11, 5632, "f16", {17: True, 33: False, 64: False}, {33: True, 49: False})])
def test_steps_of_many_rounds_keep_the_split_k_launches(hip, tmp_path, dim, heads, kvs, interm, wtype, stream_steps, prompts):
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("sg_r", 1, dim, heads, kvs, 64, seq_len=96, interm=interm), wtype, 5)
    m = hip.load_llama_model(gguf.load_gguf(str(p)), max_streams=64)
    for n, short in prompts.items():
        m.prefill([5] * n, 0, 0)
        assert short_step(m) == short, (n, "prompt")
    m.reset()
    for n, short in stream_steps.items():
        m.forward_batch(list(range(n)), [7] * n, [0] * n)
        assert short_step(m) == short, (n, "streams")
    m.close()
