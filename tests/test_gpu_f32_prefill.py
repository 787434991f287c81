"""fp32 models from 33 rows on: the matrix-core GEMM (every tile, TSHIP_F32_TILE) and the tiled prefill attention, at the edges
of their tiles, against the oracle."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu

FP32_REL = 1e-4      # the fp32 bar of the parity tests

SHAPES = {
    # hidden, heads, kv heads, ffn, attention, norm, activation; head sizes 16 / 32 / 64 / 128, one to eight query heads per KV head
    "d16_g3": (144, 9, 3, 202, synth.GQA, synth.RMSNORM, synth.SWIGLU),          # odd FFN width: rows that are not 16-byte aligned
    "d32_g5": (160, 5, 1, 72, synth.GQA, synth.LAYERNORM, synth.RELU),
    "d64_g1": (192, 3, 3, 260, synth.MHA, synth.LAYERNORM, synth.RELU),
    "d64_g7": (448, 7, 1, 96, synth.GQA, synth.RMSNORM, synth.SILU),
    "d128_g2": (512, 4, 2, 136, synth.GQA, synth.RMSNORM, synth.SWIGLU),
    "d16_g16": (256, 16, 1, 68, synth.GQA, synth.RMSNORM, synth.SILU),           # two groups of eight heads
}


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _model(shape, batch, prompt):
    hidden, heads, kv, ffn, attn, norm, act = SHAPES[shape]
    cfg = synth._cfg(n_layers=2, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=157, attn_type=attn, norm_type=norm, act=act,
                     batch=batch, prompt=prompt, steps=2, dtype="f32")
    w = synth.make_weights(cfg, 51, random_bias=True)
    for k in list(w):                                        # attention far from uniform
        if k.endswith((".Q", ".K", ".QKV")):
            w[k] = w[k] * np.float32(6.0)
    return cfg, w, synth.make_prompts(cfg, 52)


def _check(gpu, orc, lg, what):
    got = gpu.logits()
    assert np.abs(got - lg).max() <= FP32_REL * np.abs(lg).max(), what


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,prompt", [(1, 33), (3, 1), (5, 13), (1, 64), (2, 65), (3, 90), (1, 130)])
def test_prefill(G, oracle, attention, monkeypatch, shape, batch, prompt):
    cfg, w, seqs = _model(shape, batch, prompt)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 8)
    for tile in (None, "11", "21", "22", "42"):
        if tile is None:
            monkeypatch.delenv("TSHIP_F32_TILE", raising=False)
        else:
            monkeypatch.setenv("TSHIP_F32_TILE", tile)
        gpu.reset()
        gpu.prefill(seqs)
        _check(gpu, orc, lg, tile)
    gpu.close()


@pytest.fixture(params=["0", "1"], ids=["by_query", "tiles"])
def attention(request, monkeypatch):
    """Both attention kernels, whichever the rule takes."""
    monkeypatch.setenv("TSHIP_F32_ATTN", request.param)


@pytest.mark.parametrize("shape", ["d16_g3", "d64_g1", "d128_g2"])
def test_prefill_behind_a_context_and_padded(G, oracle, attention, shape):
    """A second prompt behind cached positions, and prompts padded to one length (rows that see every position)."""
    cfg, w, seqs = _model(shape, 3, 45 + 38)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=3, max_seq_len=96)
    gpu.prefill(seqs[:, :45])
    gpu.prefill(seqs[:, 45:])
    _check(gpu, orc, lg, "turn")
    lens = np.array([83, 20, 33], np.int32)
    ids, _ = G.HipGpt.pad_sentences([list(s[:n]) for s, n in zip(seqs, lens)], pad_id=0)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(ids, use_cache=True, lens=lens.astype(np.float32))
    gpu.reset()
    gpu.prefill(ids, lens=lens)
    # (a padding row's scores are rounded to 2^-9: a score on the edge of a step moves its probability by 0.2 %)
    err = np.abs(gpu.logits() - lg).max() / np.abs(lg).max()
    assert err <= 10 * FP32_REL
    gpu.close()


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("at,bad", [(37, np.inf), (64, np.nan), (89, -np.inf)])      # inside a chunk of 32 positions, its first, the prompt's last
def test_prefill_with_a_non_finite_row(G, attention, shape, at, bad):
    """A token whose key and value are not finite: the positions in front of it are those of a prompt without it, bit for bit."""
    cfg, w, seqs = _model(shape, 2, 90)
    w["TgtEmbeddings"][5] = bad
    seqs[seqs == 5] = 6
    gpu = G.HipGpt(cfg, w, max_batch=2, max_seq_len=104)

    def run(ids):
        gpu.reset()
        gpu.prefill(ids)
        return gpu.logits(), gpu.get_kv(1, 0), gpu.get_kv(1, 1)       # (the second layer's keys and values follow the first one's attention)

    want = run(seqs)
    seqs[1, at] = 5
    got = run(seqs)
    assert all(np.isfinite(x).all() for x in want) and np.array_equal(got[0][0], want[0][0])
    for a, b in zip(want[1:], got[1:]):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1, :, :at], b[1, :, :at])
        assert not np.isfinite(b[1, :, at:]).any()
    gpu.close()


@pytest.mark.parametrize("hidden,heads,kv,batch,context,tokens,tiles", [
    (64, 4, 2, 1, 400, 1, False), (64, 4, 2, 1, 400, 33, False), (512, 8, 8, 1, 400, 2, False), (256, 2, 2, 1, 0, 32, False),      # head sizes 16, 16, 64, 128
    (512, 8, 1, 1, 400, 2, True), (512, 8, 8, 4, 0, 300, True), (64, 4, 2, 16, 400, 128, True)])
def test_short_prompts_take_a_block_per_query(G, monkeypatch, hidden, heads, kv, batch, context, tokens, tiles):
    """Few tokens behind a long context with small heads, against many tokens and against eight heads on a KV head."""
    cfg = synth._cfg(n_layers=1, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=64, vocab=157, attn_type=synth.GQA, norm_type=synth.RMSNORM,
                     act=synth.RELU, batch=batch, prompt=tokens, steps=1, dtype="f32")
    gpu = G.HipGpt(cfg, synth.make_weights(cfg, 53), max_batch=batch, max_seq_len=context + tokens + 8)
    if context:
        gpu.set_seq_len(batch, context)
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    gpu.prefill(synth.make_prompts(cfg, 54))
    kernels = gpu.profile_symbols()
    assert any("attn_prefill_f32_kernel" in k for k in kernels) == tiles and any("attn_prefill_kernel" in k for k in kernels) != tiles, kernels
    gpu.close()


def test_generate_with_more_than_32_rows(G, oracle):
    """The same GEMM at decode (split K, replayed from a captured graph): 40 sequences, greedy."""
    cfg, w, seqs = _model("d64_g1", 40, 3)
    orc = oracle.OracleGpt(cfg, w)
    p, _ = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=40, max_seq_len=16)
    gpu.prefill(seqs)
    ids, _ = gpu.generate(5)
    cur = seqs
    for i in range(5):
        nxt = oracle.argmax(p).astype(np.int32)
        assert np.array_equal(ids[i], nxt), i
        cur = np.concatenate([cur, nxt[:, None]], 1)
        p, lg = orc.step(cur, use_cache=True)
    _check(gpu, orc, lg, "generate")
    gpu.close()
