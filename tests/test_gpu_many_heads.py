"""Decode steps of models with several hundred heads (caches without the fragment layout), against the oracle."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


# 255 heads and more: hidden 4080 / 16 and 8192 / 16 (the most there can be), as many KV heads or few of them
@pytest.mark.parametrize("dtype,hidden,heads,kv", [("f32", 4080, 255, 255), ("f32", 4096, 256, 256), ("f32", 4096, 256, 8), ("f16", 8192, 512, 4), ("f16", 4160, 260, 260),
                                                   ("f16", 8192, 256, 64)])
def test_steps(G, oracle, dtype, hidden, heads, kv):
    cfg = synth._cfg(n_layers=1, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=32, vocab=64, attn_type=synth.MHA if kv == heads else synth.GQA,
                     norm_type=synth.RMSNORM, act=synth.RELU, batch=1, prompt=3, steps=2, dtype=dtype)
    w = synth.make_weights(cfg, 81, random_bias=True)
    seqs = synth.make_prompts(cfg, 82)
    orc = oracle.OracleGpt(cfg, w)
    p, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=1, max_seq_len=8)
    gpu.prefill(seqs)
    for _ in range(2):
        nxt = oracle.argmax(p).astype(np.int32)
        seqs = np.concatenate([seqs, nxt[:, None]], 1)
        p, lg = orc.step(seqs, use_cache=True)
        gpu.decode(nxt)
        assert np.abs(gpu.logits() - lg).max() <= (1e-4 * np.abs(lg).max() if dtype == "f32" else 3e-2)      # (the bars of the parity tests)
    gpu.close()
