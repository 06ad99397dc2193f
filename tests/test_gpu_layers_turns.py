"""GPU: handles whose launches need the whole device, decoding from threads of their own: the ids that each gives alone, and no launch gives up
(chip_turn, nanollama_amd/csrc/nl_engine.hip)."""
import threading

import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("other", ["layers", "clusters", "persistent"])
def test_handles_take_turns(tmp_path, monkeypatch, other):
    from nanollama_amd import model as hip
    shapes = [synth.ModelShape("a", 6, 1536, 24, 6, 512, seq_len=400, interm=4096),
              {"layers": synth.ModelShape("b", 5, 1024, 16, 4, 512, seq_len=400, interm=2048),
               "clusters": synth.ModelShape("b", 5, 768, 12, 3, 512, seq_len=400, interm=2048),
               "persistent": synth.ModelShape("b", 13, 576, 9, 9, 32000, seq_len=400, interm=1536)}[other]]
    files = []
    for i, shape in enumerate(shapes):
        p = tmp_path / f"{i}.gguf"
        synth.generate_gguf(str(p), shape, "q8_0", 95 + i, mode="qrand")
        files.append(gguf.load_gguf(str(p)))

    def work(m, out):
        m.reset()
        m.prefill(list(range(3, 40)))
        out.append(m.decode_greedy(5, 37, 200))
        out.append(m.sample_decode(237, 33, temperature=0.8, top_p=0.9, top_k=50, rep_penalty=1.15, rep_window=64,
                                   uniforms=np.random.default_rng(4).random(33, dtype=np.float32), recent=[])[0])
        for i in range(20):
            m.forward(7 + i, 270 + i)
        out.append(m.state.logits.copy().tolist())

    alone = []
    for f in files:
        m, out = hip.load_llama_model(f), []
        work(m, out)
        alone.append(out)
        m.close()
    models = [hip.load_llama_model(f) for f in files]
    assert models[0].debug_read("layers_max_pos", 1)[0] > 0
    for _ in range(3):
        outs = [[] for _ in models]
        threads = [threading.Thread(target=work, args=(m, o)) for m, o in zip(models, outs)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert outs == alone
    for m in models:
        assert m.last_error() == ""
        m.close()


# one of two handles gives its launch up and goes on with the plans that wait for nobody; the other one notices nothing
def test_a_handle_that_gives_up_beside_one_that_does_not(tmp_path, monkeypatch):
    from nanollama_amd import model as hip
    shapes = [synth.ModelShape("a", 6, 1536, 24, 6, 512, seq_len=400, interm=4096), synth.ModelShape("b", 5, 1024, 16, 4, 512, seq_len=400, interm=2048)]
    files = []
    for i, shape in enumerate(shapes):
        p = tmp_path / f"{i}.gguf"
        synth.generate_gguf(str(p), shape, "q4_k", 95 + i, mode="qrand")
        files.append(gguf.load_gguf(str(p)))

    def work(m, out):
        m.reset()
        m.prefill(list(range(3, 40)))
        for k in range(6):
            out.append(m.decode_greedy(5 + k, 37 + 50 * k, 50))

    want = [[], []]
    for i, knob in ((0, "0"), (1, "1")):
        monkeypatch.setenv("NL_LAYERS", knob)
        m = hip.load_llama_model(files[i])
        work(m, want[i])
        m.close()
    monkeypatch.delenv("NL_LAYERS")
    monkeypatch.setenv("NL_QUIET", "1")
    monkeypatch.setenv("NL_FUSED_SPIN_LIMIT", "0")
    gives_up = hip.load_llama_model(files[0])
    monkeypatch.delenv("NL_FUSED_SPIN_LIMIT")
    stays = hip.load_llama_model(files[1])
    assert gives_up.layers_info()["max_pos"] == stays.layers_info()["max_pos"] == 400
    for _ in range(2):
        outs = [[], []]
        threads = [threading.Thread(target=work, args=(m, o)) for m, o in zip((gives_up, stays), outs)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert outs == want
    assert "timed out" in gives_up.last_error() and gives_up.layers_info()["max_pos"] == 0
    assert stays.last_error() == "" and stays.layers_info()["max_pos"] == 400
    third = hip.load_llama_model(files[1])                       # joins a device where one handle takes turns and one does not
    outs = [[], []]
    threads = [threading.Thread(target=work, args=(m, o)) for m, o in zip((third, stays), outs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert outs == [want[1], want[1]] and third.last_error() == stays.last_error() == ""
    for m in (gives_up, stays, third):
        m.close()
