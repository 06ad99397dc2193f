"""GPU tests of the prompt attention within one run of keys (attn_tile16_kernel, nanollama_amd/csrc/nl_batch.h): a prompt inside the first 128
positions writes the output projection's fragments from the attention launch, and leaves out key tiles and wavefronts that hold nothing.  The same
bits as partials and battn_merge_kernel (NL_NO_ATTN_FIN=1, of the same handle).  Reference: go/model.go:557-587."""
import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu

# heads, key / value heads, width: one to eight query heads a group, head sizes 32 and 64
HEADS = [(3, 3, 192), (4, 2, 256), (6, 2, 384), (8, 2, 256), (8, 1, 512), (8, 1, 256), (4, 4, 128)]


@pytest.mark.parametrize("wtype", ["q8_0", "q4_0"])
@pytest.mark.parametrize("heads,kvs,dim", HEADS)
def test_one_run_gives_the_bits_of_partials_and_merge(tmp_path, monkeypatch, heads, kvs, dim, wtype):
    from nanollama_amd import model
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("short", 2, dim, heads, kvs, 128, seq_len=192, interm=256), wtype, 29)
    m = model.load_llama_model(gguf.load_gguf(str(p)), max_streams=2)
    toks = [int(t) for t in np.random.default_rng(6).integers(3, 128, size=192)]
    for n in (8, 15, 17, 33, 63, 65, 100, 128, 129):
        got = {}
        for knob in (False, True):
            if knob:
                monkeypatch.setenv("NL_NO_ATTN_FIN", "1")
            else:
                monkeypatch.delenv("NL_NO_ATTN_FIN", raising=False)
            m.reset(0)
            m.reset(1)
            rows = []
            for at, to in ((0, n), (n, n + 11)):         # the second behind a context, across position 128 too
                m.prefill(toks[at:to], at, 1)
                rows.append(m.state.logits.copy())
                assert int(m.debug_read("step_path", 1)[0]) & 4 == (4 if to <= 128 and not knob else 0), (at, to, knob)
            got[knob] = rows
        for a, b in zip(got[False], got[True]):
            assert np.isfinite(a).all() and np.array_equal(a, b), (n, float(np.abs(a - b).max()))
    m.close()


# The projections' launch leaves K and V^T as the attention's images, or a launch of its own converts the cache: the same bits.  Token tiles of 64 and 128 (the
# last half of a chunk without a tile), one and two sets of wavefronts, 128 rows of the matrix (two heads), one to eight query heads a group; behind a
# context the images are converted.
def _images(tmp_path, monkeypatch, shape, lengths, wtype, path):
    """path: the step_path bits that every prompt from position 0 has beside the images'."""
    from nanollama_amd import model
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, wtype, 31)
    m = model.load_llama_model(gguf.load_gguf(str(p)), max_streams=2)
    toks = [int(t) for t in np.random.default_rng(7).integers(3, 128, size=max(lengths) + 300)]
    for n in lengths:
        got = {}
        for knob in (False, True):
            if knob:
                monkeypatch.setenv("NL_KV16_LAUNCH", "1")
            else:
                monkeypatch.delenv("NL_KV16_LAUNCH", raising=False)
            m.reset(0)
            m.reset(1)
            rows = []
            for at, to in ((0, n), (n, n + 290)):
                m.prefill(toks[at:to], at, 1)
                rows.append(m.state.logits.copy())
                ran = int(m.debug_read("step_path", 1)[0])
                assert ran & 16 == (16 if at == 0 and not knob else 0), (at, to, knob)
                assert at or ran & path == path, (n, ran)
            got[knob] = rows
        for a, b in zip(got[False], got[True]):
            assert np.isfinite(a).all() and np.array_equal(a, b), (n, float(np.abs(a - b).max()))
    m.close()


@pytest.mark.parametrize("wtype", ["q4_0", "q8_0", "f16"])
@pytest.mark.parametrize("heads,kvs,lengths", [(4, 2, (256, 257, 319, 320, 321, 383, 384, 385, 449)), (8, 1, (260, 300)), (6, 2, (300, 400)), (4, 4, (512, 520)),
                                               (8, 8, (1000,)), (24, 24, (1601,))])
def test_images_from_the_projections(tmp_path, monkeypatch, heads, kvs, lengths, wtype):
    monkeypatch.setenv("NL_DGEMM", "0")                   # (short Q4_0 prompts otherwise)
    _images(tmp_path, monkeypatch, synth.ModelShape("images", 2, heads * 64, heads, kvs, 128, seq_len=max(lengths) + 300, interm=256), lengths, wtype, 0)


# 513 to 1023 tiles of 64 x 64 (one set of wavefronts, 64-token tiles: 993 tokens of 24 + 6 + 6 heads are 576, 1750 of 12 + 4 + 4 560), projections with biases,
# and norms folded around the launch (Q4_0, every matrix of a layer 128 workgroups)
@pytest.mark.parametrize("wtype,heads,kvs,n,bias,fold", [("f16", 24, 6, 993, False, 0), ("q8_0", 12, 4, 1750, True, 0), ("q4_0", 24, 6, 993, False, 32),
                                                         ("q4_0", 12, 4, 1750, True, 32), ("q4_0", 24, 24, 1000, True, 32), ("f16", 4, 2, 300, True, 0)])
def test_images_from_the_projections_of_long_prompts(tmp_path, monkeypatch, wtype, heads, kvs, n, bias, fold):
    monkeypatch.setenv("NL_DGEMM", "0")
    _images(tmp_path, monkeypatch, synth.ModelShape("images", 2, heads * 64, heads, kvs, 128, seq_len=n + 300, interm=768, attn_bias=bias), (n,), wtype, fold)


# Decode batches around two workgroups a compute unit, where the attention's workgroups go from eight wavefronts to four: one split (fragments from the launch)
# and two, one to eight query heads a group (eight: always four wavefronts), heads of 32 and 64, against each stream by itself.
@pytest.mark.parametrize("head", [32, 64])
@pytest.mark.parametrize("heads,kvs,at", [(9, 9, 40), (9, 9, 130), (18, 9, 131), (36, 9, 45), (27, 9, 129), (72, 9, 140)])
def test_decode_batches_of_many_workgroups(tmp_path, heads, kvs, at, head):
    from nanollama_amd import model
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("batch", 1, heads * head, heads, kvs, 128, seq_len=192, interm=256), "q8_0", 43)
    m = model.load_llama_model(gguf.load_gguf(str(p)), max_streams=64)
    edge = 2 * int(m.debug_read("num_cus", 1)[0]) // kvs // (1 if at < 128 else 2)
    assert 1 < edge < 64
    toks = np.random.default_rng(9).integers(3, 128, size=(64, at + 1))
    for s in range(64):
        m.prefill([int(t) for t in toks[s, :at]], 0, s, want_logits=False)
    alone = []
    for s in (0, edge - 1, edge):
        m.forward(int(toks[s, at]), at, s)
        alone.append(m.state.logits.copy())
    for n in (edge, edge + 1):                             # at most two workgroups a compute unit, and more
        _, rows = m.forward_batch(list(range(n)), [int(t) for t in toks[:n, at]], [at] * n, want_logits=True)
        assert int(m.debug_read("step_path", 1)[0]) & 64 == (64 if n == edge and heads < 8 * kvs else 0), n
        for s, want in zip((0, edge - 1, edge), alone):
            if s < n:
                assert np.isfinite(rows[s]).all() and np.abs(rows[s] - want).max() <= 1e-4 * max(1.0, float(want.std())), (n, s)
    m.close()
