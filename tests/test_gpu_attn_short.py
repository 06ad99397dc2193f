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
