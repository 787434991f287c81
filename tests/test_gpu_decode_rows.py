"""Decode steps of models made for more than 32 rows (row-major GEMM tiles), at the edges of their ranges."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu

FP16_ABS = 3e-2      # the fp16 bar of the parity tests


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _cfg(hidden, heads, kv, ffn, norm, act, batch, dtype, attn=synth.GQA, prompt=5):
    return synth._cfg(n_layers=3, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=157, attn_type=attn, norm_type=norm, act=act,
                      batch=batch, prompt=prompt, steps=4, dtype=dtype)


def _steps(G, oracle, cfg, max_batch):
    w = synth.make_weights(cfg, 61, random_bias=True)
    seqs = synth.make_prompts(cfg, 62)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=max_batch, max_seq_len=24)
    p, lg = orc.step(seqs, use_cache=True)
    gpu.prefill(seqs)
    cur = seqs
    for i in range(4):
        nxt = oracle.argmax(p).astype(np.int32)
        cur = np.concatenate([cur, nxt[:, None]], 1)
        p, lg = orc.step(cur, use_cache=True)
        gpu.decode(nxt)
        assert np.abs(gpu.logits() - lg).max() <= FP16_ABS, i
    assert gpu.seq_len() == seqs.shape[1] + 4
    # the same steps from the generate loop's captured graph: same kernels, same bits
    want = gpu.logits()
    gpu.reset()
    gpu.prefill(seqs)
    ids, _ = gpu.generate(4)
    if np.array_equal(ids.T, cur[:, -4:]):       # (an fp16 model may choose another token where two are close)
        assert np.array_equal(gpu.logits(), want)
    gpu.close()


@pytest.mark.parametrize("shape", [(160, 10, 5, 200, synth.SWIGLU), (48, 3, 1, 104, synth.RELU), (512, 8, 2, 704, synth.SILU), (256, 2, 2, 96, synth.SWIGLU_SILU)])
@pytest.mark.parametrize("max_batch,batch", [(33, 33), (64, 1), (64, 64), (100, 65), (128, 128)])
def test_rows(G, oracle, shape, max_batch, batch):
    hidden, heads, kv, ffn, act = shape
    _steps(G, oracle, _cfg(hidden, heads, kv, ffn, synth.RMSNORM, act, batch, "f16"), max_batch)
