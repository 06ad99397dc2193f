"""GPU: prompts and streams of files with K-quant matrices keep the range and the precision of their single-token steps (pgemm_kernel, PG_EXACT)."""
from dataclasses import replace

import numpy as np
import pytest

from nanollama_amd import gguf, synth

pytestmark = pytest.mark.gpu
AT = {"q4_0": [0], "q8_0": [0], "q4_k": [0, 2], "q6_k": [208]}        # a block's fp16 scales
SIZE = {"q4_0": 18, "q8_0": 34, "q4_k": 144, "q6_k": 210}


class Edited:
    """A parsed file whose tensors are drawn anew in other formats and whose scales or gains are multiplied (exactly, by powers of two)."""

    def __init__(self, g, shape, types, factors=()):
        self.meta, self.tensor_order, self.raw = g.meta, g.tensor_order, {}
        for ckpt, name, tshape, kind in synth.tensor_plan(shape):
            data, info = g.get_tensor(name)
            factor = next((f for part, f in dict(factors).items() if part in name), 1.0)
            if kind in ("norm", "bias"):
                self.raw[name] = (data.view(np.float32) * np.float32(factor)).view(np.uint8), info
                continue
            t = next((v for part, v in types.items() if part in name), types["default"])
            data = synth._draw_qrand(shape, 77, ckpt, tshape, kind, synth.WTYPES[t])
            blocks = data.reshape(-1, SIZE[t])
            for at in AT[t]:
                d = (blocks[:, at:at + 2].copy().view(np.float16) * np.float32(factor)).astype(np.float16)
                assert np.isfinite(d).all()
                blocks[:, at:at + 2] = d.view(np.uint8)
            self.raw[name] = data, replace(info, type=synth.WTYPES[t])

    def get_tensor(self, name):
        return self.raw[name]


def exact_logits(orc, g, shape, toks):
    """The last token's logits in 64 bits."""
    def w(name):
        data, info = g.get_tensor(name)
        if info.type == gguf.GGML_F32:
            return data.view(np.float32).astype(np.float64)
        return orc.dequant(np.ascontiguousarray(data), info.type, info.nel).astype(np.float64).reshape(info.dims[1], info.dims[0])
    norm = lambda x, gain: x / np.sqrt((x * x).mean(-1, keepdims=True) + float(np.float32(shape.eps))) * gain
    n, hd, H, G = len(toks), shape.head_dim, shape.n_head, shape.n_kv_head
    x = w("token_embd.weight")[toks]
    angle = np.arange(n)[:, None] * shape.rope_theta ** (-np.arange(0, hd, 2) / hd)
    c, s = np.cos(angle)[:, None], np.sin(angle)[:, None]
    turn = lambda a: np.concatenate([a[..., :hd // 2] * c - a[..., hd // 2:] * s, a[..., :hd // 2] * s + a[..., hd // 2:] * c], -1)
    for i in range(shape.n_layer):
        p = f"blk.{i}."
        h = norm(x, w(p + "attn_norm.weight"))
        q, k, v = [(h @ w(p + f"attn_{m}.weight").T).reshape(n, -1, hd) for m in "qkv"]
        q, k, out = turn(q), turn(k), np.empty((n, H, hd))
        for j in range(H):
            z = np.where(np.tril(np.ones((n, n), bool)), q[:, j] @ k[:, j * G // H].T / np.sqrt(hd), -np.inf)
            z = np.exp(z - z.max(-1, keepdims=True))
            out[:, j] = z / z.sum(-1, keepdims=True) @ v[:, j * G // H]
        x = x + out.reshape(n, -1) @ w(p + "attn_output.weight").T
        h = norm(x, w(p + "ffn_norm.weight"))
        gate = h @ w(p + "ffn_gate.weight").T
        x = x + (gate / (1 + np.exp(-gate)) * (h @ w(p + "ffn_up.weight").T)) @ w(p + "ffn_down.weight").T
    return norm(x[-1], w("output_norm.weight")) @ w("output.weight").T


def errors(tmp_path, monkeypatch, shape, types, factors, prompts, first=None):
    """Relative errors against 64 bits, their root mean square over the prompts: a prompt in two portions, and token by token."""
    from nanollama_amd import model as hip
    from oracle import oracle as orc
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), shape, "q4_0", 77, mode="qrand")
    g = Edited(gguf.load_gguf(str(p)), shape, types, factors)
    with np.errstate(over="ignore"):
        want = [exact_logits(orc, g, shape, toks) for toks in prompts]
    assert np.isfinite(want).all()
    out = []
    for single in (False, True):
        if single:
            monkeypatch.setenv("NL_NO_BATCH_PATH", "1")
        dev, err = hip.load_llama_model(g), []
        for toks, w in zip(prompts, want):
            dev.reset()
            k = first or len(toks) // 2
            dev.prefill(toks[:k], want_logits=False)
            dev.prefill(toks[k:], k)
            assert np.isfinite(dev.state.logits).all(), (single, factors)
            err.append(np.linalg.norm(dev.state.logits - w) / np.linalg.norm(w))
        out.append(float(np.sqrt(np.mean(np.square(err)))))
        dev.close()
    print(f"\n{types} {dict(factors)}: prompts {out[0]:.3g}, by token {out[1]:.3g}, ratio {out[0] / out[1]:.2f}")
    return out


SHAPE = synth.ModelShape("kquant", 2, 512, 8, 2, 512, seq_len=256, interm=768)
# activations where trained models have them: feed-forward ones of 1e-4 and 1e6, attention outputs of 1e-4, values beyond what 16 bits hold
RANGES = {"as_is": (), "feed_forward_small": (("ffn_norm", 2.0 ** -7), ("ffn_down", 2.0 ** 13)), "feed_forward_large": (("ffn_norm", 2.0 ** 10),),
          "attention_small": (("attn_norm", 2.0 ** -10), ("attn_output", 2.0 ** 10)), "values_large": (("attn_v", 2.0 ** 17),)}
ALL = {"q4_k": {"default": "q4_k"}, "q6_k": {"default": "q6_k"}, "q4_k_q6_k": {"default": "q4_k", "ffn_down": "q6_k", "output.weight": "q6_k"},
       "q4_0_head_q6_k": {"default": "q4_0", "output.weight": "q6_k"}, "q4_k_ffn_q8_0": {"default": "q4_k", "ffn_": "q8_0"}}


# Not above the single-token plan's error: 0.85 - 0.97 of it on 24 prompts; a quarter more is what the mean of a few prompts varies by.
# (Activations held in fewer bits are further off: as hi + lo of 16 bits by a factor of ten to forty at 1e-4, and infinite at 1e6.)
@pytest.mark.parametrize("ranges", RANGES)
@pytest.mark.parametrize("types", ALL)
def test_prompts_are_as_exact_as_the_single_token_plan(tmp_path, monkeypatch, types, ranges):
    prompts, single = errors(tmp_path, monkeypatch, SHAPE, ALL[types], RANGES[ranges], [synth.prompt_ids(90 + 9 * i, 512, seed=i) for i in range(12)])
    assert prompts <= 1.25 * single


# every matrix on one set of wavefronts (more than 256 tiles of 64 x 64) and on two
@pytest.mark.parametrize("types", ["q4_k", "q6_k", "q4_0_head_q6_k", "q4_k_ffn_q8_0"])
def test_large_grids(tmp_path, monkeypatch, types):
    shape = synth.ModelShape("kquant_large", 2, 1024, 16, 4, 512, seq_len=1700, interm=1280)
    prompts, single = errors(tmp_path, monkeypatch, shape, ALL[types], (), [synth.prompt_ids(n, 512, seed=n) for n in (1100, 1250, 1130)], 30)
    assert prompts <= 1.5 * single        # (three prompts only)


# rows that fill no 64-row workgroup (heads of 32, 8 + 2 of them: 20 row tiles, a vocabulary of 520), biases, conjugate rotation, QK-norm
@pytest.mark.parametrize("kind", ["q4_k", "q6_k"])
@pytest.mark.parametrize("variant", ["bias_conj", "qk_norm"])
@pytest.mark.parametrize("n", [5, 64, 133])
def test_variants_against_the_oracle(tmp_path, kind, variant, n):
    from nanollama_amd import model as hip
    from oracle import oracle as orc
    shape = synth.ModelShape("kquant_v", 2, 256, 8, 1, 520, seq_len=160, interm=768, attn_bias=variant == "bias_conj", rope_conjugate=variant == "bias_conj", qk_norm=variant == "qk_norm")
    p = tmp_path / "v.gguf"
    synth.generate_gguf(str(p), shape, kind, 37)
    g = gguf.load_gguf(str(p))
    toks = synth.prompt_ids(n, shape.vocab, seed=8)
    ref, dev = orc.OracleModel(g), hip.load_llama_model(g)
    for pos, t in enumerate(toks):
        want = ref.forward(t, pos)
    dev.prefill(toks)
    assert np.abs(dev.state.logits - want).max() <= 1e-4 * max(1.0, float(want.std()))
    nxt = int(np.argmax(want))
    assert dev.decode_greedy(nxt, n, 3)[0] == int(np.argmax(ref.forward(nxt, n)))
    dev.close()


def test_streams_are_as_exact_as_the_single_token_plan(tmp_path, monkeypatch):
    from nanollama_amd import model as hip
    from oracle import oracle as orc
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), SHAPE, "q4_0", 77, mode="qrand")
    g = Edited(gguf.load_gguf(str(p)), SHAPE, ALL["q4_k"], RANGES["feed_forward_large"])
    toks = [synth.prompt_ids(20 + 11 * s, 512, seed=s) for s in range(12)]
    want = [exact_logits(orc, g, SHAPE, t) for t in toks]
    rel = lambda a: [np.linalg.norm(x - y) / np.linalg.norm(y) for x, y in zip(a, want)]
    err = []
    for single in (False, True):
        if single:
            monkeypatch.setenv("NL_NO_BATCH_PATH", "1")
        dev = hip.load_llama_model(g, max_streams=12)
        for s, t in enumerate(toks):
            dev.prefill(t[:-1], 0, s, want_logits=False)
        _, rows = dev.forward_batch(list(range(12)), [t[-1] for t in toks], [len(t) - 1 for t in toks], want_logits=True)
        err.append(float(np.sqrt(np.mean(np.square(rel(rows))))))
        dev.close()
    print(f"\nstreams {err[0]:.3g}, one by one {err[1]:.3g}")
    assert err[0] <= 1.25 * err[1]


@pytest.mark.parametrize("kind", ["q4_k", "q6_k"])
def test_few_tokens_run_the_single_token_plan(tmp_path, kind):
    # (below five tokens a multi-token step costs more than the single-token ones: the same bits)
    from nanollama_amd import model as hip
    p = tmp_path / "m.gguf"
    synth.generate_gguf(str(p), SHAPE, kind, 19)
    dev = hip.load_llama_model(gguf.load_gguf(str(p)), max_streams=5)
    for n in (3, 4, 5):
        dev.prefill(list(range(7, 7 + n)))
        got = dev.state.logits.copy()
        dev.reset()
        for i in range(n):
            dev.forward(7 + i, i)
        assert np.array_equal(got, dev.state.logits) == (n < 5), n
        _, rows = dev.forward_batch(list(range(n)), [40 + s for s in range(n)], [0] * n, want_logits=True)
        one = []
        for s in range(n):
            dev.forward(40 + s, 0, s)
            one.append(dev.state.logits.copy())
        assert np.array_equal(rows, one) == (n < 5), n
    dev.close()
