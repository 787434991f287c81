"""The bar of the fp16 parity tests on tiny models against what it has to catch: on the oracle, a projection of any one layer
that returns zero moves the logits by several times the bar, at the prompt and at a cached step."""
import numpy as np
import pytest

from parity_util import FP16_SENSITIVE_REL, sensitive
from seq2seqsharp_amd import synth
from test_gpu_decode_rows import SHAPES as STEP_SHAPES
from test_gpu_decode_rows import SPLIT_SHAPES
from test_gpu_decode_rows import _cfg
from test_gpu_prefill_tiles import SHAPES as TILE_SHAPES

MODELS = {"step%d" % i: (h, n, kv, ffn, synth.RMSNORM, act, synth.GQA) for i, (h, n, kv, ffn, act) in enumerate(STEP_SHAPES)}
MODELS.update({"split%d" % i: s + (synth.GQA,) for i, s in enumerate(SPLIT_SHAPES)})
MODELS.update({name: (h, n, kv, ffn, norm, act, attn) for name, (h, n, kv, ffn, attn, norm, act) in TILE_SHAPES.items()})


@pytest.mark.parametrize("name", sorted(MODELS))
def test_a_projection_that_returns_zero_is_beyond_the_bar(oracle, name):
    hidden, heads, kv, ffn, norm, act, attn = MODELS[name]
    cfg = _cfg(hidden, heads, kv, ffn, norm, act, 4, "f16", attn=attn)
    w = sensitive(synth.make_weights(cfg, 61, random_bias=True), hidden)
    seqs = synth.make_prompts(cfg, 62)

    def logits(w):
        orc = oracle.OracleGpt(cfg, w)
        return orc.step(seqs, use_cache=True)[1], orc.step(np.concatenate([seqs, seqs[:, :1]], 1), use_cache=True)[1]

    want = logits(w)
    parts = []
    for layer in range(cfg["n_layers"]):
        a, f = "GPTDecoder.SelfAttn_%d" % layer, "GPTDecoder.PosFFN_%d.feedForwardLayer" % layer
        parts += [(n, slice(None)) for n in [a + s for s in (".Q", ".K", ".V", ".W0")] + [f + s for s in ("1.m_Whd", "2.m_Whd", "3.m_Whd")] if n in w]
        parts += [(a + ".QKV", slice(i * hidden, (i + 1) * hidden)) for i in range(3) if a + ".QKV" in w]
    assert len(parts) >= 6 * cfg["n_layers"]
    for n, cols in parts:
        broken = w[n].copy()
        broken[:, cols] = 0.0
        for a, b in zip(want, logits(dict(w, **{n: broken}))):
            assert np.abs(a - b).max() > 5 * FP16_SENSITIVE_REL * np.abs(a).max(), n
