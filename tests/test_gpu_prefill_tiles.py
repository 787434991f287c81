"""Every tile of the prefill GEMMs (TSHIP_GEMM_TILE) at the edges of its range, against the oracle."""
import numpy as np
import pytest

from parity_util import FP16_SENSITIVE_REL, sensitive
from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu

FP16_ABS = 3e-2      # the fp16 bar of the parity tests

SHAPES = {
    # hidden, heads, kv heads, ffn, attention, norm, activation; k-tiles of 16: 10 / 12.5 (a partial last one), 3 / 7, 32 / 44
    "rms_gated": (160, 10, 5, 200, synth.GQA, synth.RMSNORM, synth.SWIGLU),
    "layer_norm_relu": (48, 3, 3, 104, synth.MHA, synth.LAYERNORM, synth.RELU),
    "rms_silu_wide": (512, 8, 2, 704, synth.GQA, synth.RMSNORM, synth.SILU),
}


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _model(shape, batch, prompt):
    hidden, heads, kv, ffn, attn, norm, act = SHAPES[shape]
    cfg = synth._cfg(n_layers=2, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=157, attn_type=attn, norm_type=norm, act=act,
                     batch=batch, prompt=prompt, steps=2, dtype="f16")
    return cfg, sensitive(synth.make_weights(cfg, 41, random_bias=True), hidden), synth.make_prompts(cfg, 42)


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,prompt", [(1, 1), (1, 33), (1, 64), (5, 13), (2, 65), (3, 90), (5, 128)])      # 1 ... 640 rows around 64, 128 and 256
def test_prefill_gemm_tiles(G, oracle, monkeypatch, shape, batch, prompt):
    """Logits, keys and values with each tile; one row, rows that end inside, at and behind a 64-row group, column counts that
    are no multiple of a tile's columns, k-tile counts that are no multiple of a stage's.  Tile 0 applies from 256 rows on."""
    cfg, w, seqs = _model(shape, batch, prompt)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 8)
    for tile in (None, "11", "12", "14", "22", "24", "0"):
        if tile is None:
            monkeypatch.delenv("TSHIP_GEMM_TILE", raising=False)
        else:
            monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
        gpu.reset()
        gpu.prefill(seqs)
        got = gpu.logits()
        assert np.abs(got - lg).max() <= FP16_SENSITIVE_REL * np.abs(lg).max(), tile
        k, v = gpu.get_kv(1, 0), gpu.get_kv(1, 1)
        if tile is None:
            k0, v0 = k, v
        # one fp16 rounding step of the stored value (2^-10 of it) and the same of the sums in front of it, in another order
        assert np.abs(k - k0).max() <= 4e-3 * np.abs(k0).max() and np.abs(v - v0).max() <= 4e-3 * np.abs(v0).max(), tile
    gpu.close()


@pytest.mark.parametrize("hidden,heads,kv,batch,prompt", [(512, 8, 2, 5, 128), (1024, 8, 2, 3, 192), (512, 8, 4, 1, 544)])
def test_large_tile_writes_whole_fragments_like_pieces(G, monkeypatch, hidden, heads, kv, batch, prompt):
    """The 256 x 256 tile forced: whole fragments of the cache (head sizes 64 and 128, a wavefront partly beyond the
    rows) against pieces, and the heights of the tile patches against each other, bit for bit."""
    cfg = synth._cfg(n_layers=2, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=2 * hidden, vocab=157, attn_type=synth.GQA,
                     norm_type=synth.RMSNORM, act=synth.SWIGLU, batch=batch, prompt=prompt, steps=2, dtype="f16")
    w = synth.make_weights(cfg, 77, random_bias=True)
    seqs = synth.make_prompts(cfg, 78)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 8)
    monkeypatch.setenv("TSHIP_GEMM_TILE", "0")
    gpu.prefill(seqs)
    want = [gpu.logits()] + [gpu.get_kv(l, i) for l in range(2) for i in range(2)]
    for name, value in (("TSHIP_NO_KV_FUSE", "1"), ("TSHIP_PATCH_ROWS", "1"), ("TSHIP_PATCH_ROWS", "8")):
        monkeypatch.setenv(name, value)
        gpu.reset()
        gpu.prefill(seqs)
        monkeypatch.delenv(name)
        got = [gpu.logits()] + [gpu.get_kv(l, i) for l in range(2) for i in range(2)]
        assert all(np.array_equal(a, b) for a, b in zip(want, got)), (name, value)
    gpu.close()


@pytest.mark.parametrize("batch,prompt", [(1, 33), (3, 90), (7, 73)])       # up to 511 rows
def test_short_prompts_keep_large_residuals(G, oracle, batch, prompt):
    """A first token whose residual, times the norms' gain, is beyond the fp16 range: rows of a short prompt are normalised
    before they are stored in 16 bits."""
    cfg, w, seqs = _model("rms_gated", batch, prompt)
    w["TgtEmbeddings"][5] = np.float16(2e4) * np.sign(w["TgtEmbeddings"][5])      # x sqrt(160): a residual of 2.5e5
    seqs[seqs == 5] = 6
    seqs[:, 0] = 5
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 8)
    gpu.prefill(seqs)
    got = gpu.logits()
    assert np.isfinite(got).all() and np.abs(got - lg).max() <= FP16_ABS
    gpu.close()


@pytest.mark.parametrize("norm,act", [(synth.RMSNORM, synth.SWIGLU), (synth.LAYERNORM, synth.RELU)])
@pytest.mark.parametrize("batch,prompt", [(5, 300), (4, 549)])       # QKV and up, and output and down, in two launches
def test_columns_in_two_launches(G, monkeypatch, norm, act, batch, prompt):
    """Projections whose columns are taken by two launches of different tiles, against one tile for all of them: keys and values
    of the second layer stand on every row and column of the first one's projections."""
    ffn = 5632 if act == synth.SWIGLU else 11264
    cfg = synth._cfg(n_layers=2, hidden=2048, n_heads=32, n_kv_heads=8, ffn_dim=ffn, vocab=157, attn_type=synth.GQA, norm_type=norm, act=act,
                     batch=batch, prompt=prompt, steps=2, dtype="f16")
    w = synth.make_weights(cfg, 91, random_bias=True)
    seqs = synth.make_prompts(cfg, 92)
    monkeypatch.setenv("TSHIP_ALL_ROWS", "1")
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 8)
    got = []
    for tile in (None, "24"):
        if tile:
            monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
        gpu.reset()
        gpu.prefill(seqs)
        n = sum("gemm" in s for s in gpu.profile_symbols())
        got.append((n, gpu.logits(), gpu.get_kv(1, 0), gpu.get_kv(1, 1)))
    gpu.close()
    assert got[1][0] == 4 * 2 + 1 and got[0][0] >= 6 * 2 + 1
    assert np.abs(got[0][1] - got[1][1]).max() <= FP16_SENSITIVE_REL * np.abs(got[1][1]).max()
    for a, b in zip(got[0][2:], got[1][2:]):      # (fp16 steps of the values and of the sums in front of them, in another order)
        assert np.abs(a - b).max() <= 4e-3 * np.abs(b).max()
