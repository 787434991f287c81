"""Decode projections of fp16 models whose wavefronts request their fragments in batches of two, four or eight, whole and partly
beyond the k range, and tails of few splits: against the oracle."""
import numpy as np
import pytest

from parity_util import FP16_SENSITIVE_REL, sensitive
from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


# hidden -> fragments per wavefront of the vocabulary projection: 4, 5, 6, 7, 11 (and half of that or more splits elsewhere)
@pytest.mark.parametrize("hidden,heads,kv,ffn", [(512, 8, 2, 832), (640, 10, 5, 448), (768, 12, 12, 3072), (896, 14, 2, 576), (1408, 11, 11, 256),
                                                   # few column tiles: tails of one, two and eight splits, ranges of uneven length
                                                   (128, 2, 2, 2048), (256, 4, 2, 1072), (352, 11, 1, 32)])
@pytest.mark.parametrize("norm,act", [(synth.RMSNORM, synth.SWIGLU), (synth.LAYERNORM, synth.RELU)])
@pytest.mark.parametrize("max_batch,batch", [(1, 1), (32, 17), (64, 33), (128, 65)])
def test_steps(G, oracle, hidden, heads, kv, ffn, norm, act, max_batch, batch):
    cfg = synth._cfg(n_layers=1, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=157, attn_type=synth.GQA, norm_type=norm, act=act,
                     batch=batch, prompt=3, steps=4, dtype="f16")
    w = sensitive(synth.make_weights(cfg, 101, random_bias=True), hidden)
    seqs = synth.make_prompts(cfg, 102)
    orc = oracle.OracleGpt(cfg, w)
    p, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=max_batch, max_seq_len=16)
    gpu.prefill(seqs)
    assert np.abs(gpu.logits() - lg).max() <= FP16_SENSITIVE_REL * np.abs(lg).max()
    for _ in range(2):
        nxt = oracle.argmax(p).astype(np.int32)
        seqs = np.concatenate([seqs, nxt[:, None]], 1)
        p, lg = orc.step(seqs, use_cache=True)
        gpu.decode(nxt)
        assert np.abs(gpu.logits() - lg).max() <= FP16_SENSITIVE_REL * np.abs(lg).max()
    gpu.close()
