"""GPU: the float32 prompt attention of K-quant files (attn_tile_kernel, nanollama_amd/csrc/nl_batch.h): a prompt inside the first 128 positions writes the
output projection's fragments from the attention launch, the same bits as partials and battn_merge_kernel (NL_NO_ATTN_FIN=1), key tiles that no row sees
are left out, and small grids share a tile of rows among a workgroup's wavefronts (attn_rows_kernel; NL_ATTN_ROWS=0: never), the same bits again.  Reference: go/model.go:557-587."""
import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu

# heads, key / value heads, width: one to eight query heads a group, head sizes 32 and 64, rows that fill no whole tile
HEADS = [(12, 4, 768), (8, 4, 256), (8, 2, 512), (8, 1, 512), (16, 2, 512), (4, 4, 256)]


@pytest.mark.parametrize("wtype", ["q4_k", "q6_k"])
@pytest.mark.parametrize("heads,kvs,dim", HEADS)
def test_one_split_gives_the_bits_of_partials_and_merge(tmp_path, monkeypatch, heads, kvs, dim, wtype):
    from nanollama_amd import model
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("exact", 2, dim, heads, kvs, 256, seq_len=192, interm=256), wtype, 31)
    m = model.load_llama_model(gguf.load_gguf(str(p)), max_streams=2)
    toks = [int(t) for t in np.random.default_rng(8).integers(3, 256, size=192)]
    for n in (8, 16, 17, 32, 33, 63, 65, 97, 128, 129):
        got = {}
        for knob, rows_too in ((False, True), (True, True), (False, False), (True, False)):
            if knob:
                monkeypatch.setenv("NL_NO_ATTN_FIN", "1")
            else:
                monkeypatch.delenv("NL_NO_ATTN_FIN", raising=False)
            monkeypatch.setenv("NL_ATTN_ROWS", "1" if rows_too else "0")
            m.reset(0)
            m.reset(1)
            rows = []
            for at, to in ((0, n), (n, n + 11)):         # the second behind a context, across position 128 too
                m.prefill(toks[at:to], at, 1)
                rows.append(m.state.logits.copy())
                assert int(m.debug_read("step_path", 1)[0]) & 132 == (4 if to <= 128 and not knob else 0) + (128 if rows_too else 0), (at, to, knob)
            got[knob, rows_too] = rows
        for other in ((True, True), (False, False), (True, False)):
            for a, b in zip(got[False, True], got[other]):
                assert np.isfinite(a).all() and np.array_equal(a, b), (n, other, float(np.abs(a - b).max()))
        if n <= 33:      # the same rows one token at a time (the per-token attention; float32 sums in another order through two layers)
            m.reset(0)
            for i, t in enumerate(toks[:n]):
                m.forward(t, i, 0)
            assert np.abs(m.state.logits - got[False, True][0]).max() <= 1e-4 * max(1.0, float(got[False, True][0].std())), n
    m.close()


@pytest.mark.parametrize("n,at,rows", [(444, 0, True), (445, 0, False), (256, 300, True), (264, 300, False)])
def test_grids_on_both_sides_of_the_rule(tmp_path, monkeypatch, n, at, rows):
    from nanollama_amd import model
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), synth.ModelShape("rule", 1, 512, 8, 2, 256, seq_len=576, interm=256), "q4_k", 33)
    m = model.load_llama_model(gguf.load_gguf(str(p)))
    toks = [int(t) for t in np.random.default_rng(9).integers(3, 256, size=576)]
    got = []
    for knob in ("1", "0"):
        monkeypatch.setenv("NL_ATTN_ROWS", knob)
        m.reset()
        if at:
            m.prefill(toks[:at], 0)
        m.prefill(toks[at:at + n], at)
        assert int(m.debug_read("step_path", 1)[0]) & 128 == (128 if rows and knob == "1" else 0)
        got.append(m.state.logits.copy())
    assert np.isfinite(got[0]).all() and np.array_equal(*got)
    m.close()
