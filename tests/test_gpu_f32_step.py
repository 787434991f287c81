"""Decode steps of dense fp32 models (five launches per layer): rows, splits of K, column tiles and head sizes at the edges of
their ranges, against the oracle."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu

FP32_REL = 1e-4      # the fp32 bar of the parity tests

SHAPES = {
    # hidden, heads, kv heads, ffn, vocab, attention, norm, activation
    "one_tile": (32, 2, 1, 32, 31, synth.GQA, synth.RMSNORM, synth.SWIGLU),              # a single tile of 32 columns, fewer tokens than that
    "d128_ln": (256, 2, 2, 96, 157, synth.MHA, synth.LAYERNORM, synth.RELU),             # vocabulary rows that are not 16-byte aligned
    "split": (416, 13, 13, 1184, 1000, synth.MHA, synth.LAYERNORM, synth.SILU),          # K splits that are no multiple of a batch
    "gated": (512, 8, 2, 1056, 352, synth.GQA, synth.RMSNORM, synth.SWIGLU_SILU),
    "wide": (2048, 32, 4, 64, 96, synth.GQA, synth.RMSNORM, synth.LEAKYRELU),            # the most columns whose statistics a block combines
    "d16_g16": (256, 16, 1, 64, 64, synth.GQA, synth.RMSNORM, synth.SILU),               # two groups of eight heads
}


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _cfg(shape, batch, **kw):
    hidden, heads, kv, ffn, vocab, attn, norm, act = shape
    return synth._cfg(n_layers=2, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=vocab, attn_type=attn, norm_type=norm, act=act,
                      batch=batch, prompt=5, steps=4, dtype="f32", **kw)


@pytest.mark.parametrize("batch", [1, 2, 3, 8, 9, 17, 32])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_steps(G, oracle, name, batch):
    """Steps behind a prompt against the oracle; the generate loop (captured) and a second pass give the same bits."""
    cfg = _cfg(SHAPES[name], batch)
    w = synth.make_weights(cfg, 71, random_bias=True)
    w["TgtEmbeddings"] = w["TgtEmbeddings"] + np.float32(0.05)          # rows whose mean is not small against their spread
    seqs = synth.make_prompts(cfg, 72)
    orc = oracle.OracleGpt(cfg, w)
    p, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=16)
    gpu.prefill(seqs)
    cur, got = seqs, []
    for _ in range(3):
        nxt = oracle.argmax(p).astype(np.int32)
        cur = np.concatenate([cur, nxt[:, None]], 1)
        p, lg = orc.step(cur, use_cache=True)
        gpu.decode(nxt)
        got.append(gpu.logits())
        assert np.abs(got[-1] - lg).max() <= FP32_REL * np.abs(lg).max()
    for _ in range(2):
        gpu.set_seq_len(batch, 5)
        gpu.decode(cur[:, 5])
        assert np.array_equal(gpu.logits(), got[0])
        ids, _ = gpu.generate(2)
        assert np.array_equal(ids.reshape(2, batch), cur[:, 6:8].T) and np.array_equal(gpu.logits(), got[2])
    gpu.close()


def test_first_position_and_the_kernels_that_run(G, oracle):
    """A step on an empty cache; five launches a layer, and the general path for a hidden size that is no multiple of 32."""
    for hidden, fused in ((96, True), (48, False)):
        cfg = _cfg((hidden, 3, 3, 64, 157, synth.MHA, synth.LAYERNORM, synth.RELU), 2)
        w = synth.make_weights(cfg, 73, random_bias=True)
        first = synth.make_prompts(cfg, 74)[:, :1]
        _, lg = oracle.OracleGpt(cfg, w).step(first, use_cache=True)
        gpu = G.HipGpt(cfg, w, max_batch=2, max_seq_len=8)
        gpu.decode(first[:, 0])
        assert np.abs(gpu.logits() - lg).max() <= FP32_REL * np.abs(lg).max()
        names = [n for n, _ in gpu.profile_decode(first[:, 0])]
        symbols = gpu.profile_symbols()
        assert any("step_gemm_f32_kernel" in s for s in symbols) == fused
        assert (len(names) == 2 + 5 * cfg["n_layers"]) == fused
        gpu.close()
