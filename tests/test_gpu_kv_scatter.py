"""The QKV projection of an fp16 prefill writing the fragment-major cache in pieces."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


# hidden, heads, kv heads, norm: head sizes 64 and 128; key columns that begin inside a tile of 64 to 320 columns
SHAPES = {"d64_gqa": (512, 8, 2, synth.RMSNORM), "d64_mha": (192, 3, 3, synth.LAYERNORM), "d128": (384, 3, 1, synth.RMSNORM)}


def _model(shape, batch, length):
    hidden, heads, kv, norm = SHAPES[shape]
    cfg = synth._cfg(n_layers=2, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=192, vocab=157, attn_type=synth.GQA, norm_type=norm, act=synth.RELU,
                     batch=batch, prompt=length, steps=2, dtype="f16")
    return cfg, synth.make_weights(cfg, 111, random_bias=True), synth.make_prompts(cfg, 112)


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,prompt,context", [(1, 1, 0), (1, 31, 0), (2, 33, 0), (3, 65, 20), (2, 40, 32), (5, 128, 0), (1, 700, 0), (9, 5, 7)])
def test_cache_in_pieces(G, oracle, monkeypatch, shape, batch, prompt, context):
    """Prompts that end inside and at 32-position chunks, shorter than a chunk's rest, behind a context; every kind of tile, whole and
    partly beyond the matrix: the cache against the oracle's, and over one that a longer prompt has filled the bits of a new model's, two steps
    behind it included."""
    hidden, heads, kv, _ = SHAPES[shape]
    total, d = context + prompt, hidden // heads
    cfg, w, seqs = _model(shape, batch, total)
    longer = np.random.default_rng(113).integers(4, 157, size=(batch, total + 40)).astype(np.int32)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    want = []
    for l in range(2):
        want.append(orc.get_cache(l, 0).reshape(batch, heads, d, total)[:, ::heads // kv].transpose(0, 1, 3, 2))
        want.append(orc.get_cache(l, 1).reshape(batch, heads, total, d)[:, ::heads // kv])
    used = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=total + 48)
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    for tile in (None, "0", "11", "14", "222", "24", "42", "43", "45"):
        if tile:
            monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
        got = []
        new = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=total + 48)
        for gpu in (used, new):
            if gpu is used:
                gpu.reset()
                gpu.prefill(longer)
                gpu.reset()
            if context:
                gpu.prefill(seqs[:, :context])
            gpu.prefill(seqs[:, context:])
            assert not any("kv_write" in s for s in gpu.profile_symbols())
            out = [gpu.logits()] + [gpu.get_kv(l, i) for l in range(2) for i in range(2)]
            for _ in range(2):
                gpu.decode((np.arange(batch) + 5).astype(np.int32))
                out.append(gpu.logits())
            got.append(out)
        new.close()
        for a, b in zip(*got):
            assert np.array_equal(a, b), tile
        assert np.abs(got[0][0] - lg).max() <= 3e-2        # (the fp16 bar of the parity tests)
        for a, b in zip(got[0][1:5], want):                # fp16 activations in front of the projection and one rounding of its output, 2^-11 of a value each
            assert np.abs(a - b).max() <= 1e-2 * np.abs(b).max(), tile
    used.close()


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,prompt,context", [(5, 70, 0), (5, 65, 20), (7, 40, 5), (1, 700, 0), (3, 333, 0), (5, 96, 0)])
def test_pieces_are_the_bits_of_whole_fragments(G, monkeypatch, shape, batch, prompt, context):
    """Keys and values of the first layer follow from each token alone, and every width of the 256-row tile adds a sum in the same order: a
    prompt's are those of the same tokens at the front of one in whole 32-position chunks, which the 256 x 256 tile writes as whole
    fragments.  (256 rows or more, and both prompts below 512 or neither: from there on the norm is deferred.)"""
    total = context + prompt
    whole = -(-total // 32) * 32
    assert batch * prompt >= 256 and (batch * whole >= 512) == (batch * prompt >= 512)
    cfg, w, seqs = _model(shape, batch, whole)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=whole + 8)
    monkeypatch.setenv("TSHIP_GEMM_TILE", "0")
    gpu.prefill(seqs)
    want = [gpu.get_kv(0, i)[:, :, context:total] for i in range(2)]
    monkeypatch.setenv("TSHIP_NO_KV_FUSE", "1")
    for tile in ("0", "42", "43", "45"):
        monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
        gpu.reset()
        if context:
            gpu.prefill(seqs[:, :context])
        gpu.prefill(seqs[:, context:total])
        for i in range(2):
            assert np.array_equal(gpu.get_kv(0, i)[:, :, context:], want[i]), tile
    gpu.close()
