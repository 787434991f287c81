"""Decode steps of models made for more than 32 rows (row-major GEMM tiles) and the in-place move of cache rows, at the edges
of their ranges."""
import numpy as np
import pytest

from parity_util import FP16_SENSITIVE_REL, sensitive
from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu

# hidden, heads, kv heads, ffn, activation
SHAPES = [(160, 10, 5, 200, synth.SWIGLU), (48, 3, 1, 104, synth.RELU), (512, 8, 2, 704, synth.SILU), (256, 2, 2, 96, synth.SWIGLU_SILU)]
SPLIT_SHAPES = [(160, 10, 5, 1000, synth.RMSNORM, synth.SWIGLU), (512, 8, 2, 704, synth.LAYERNORM, synth.RELU)]


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _cfg(hidden, heads, kv, ffn, norm, act, batch, dtype, attn=synth.GQA, prompt=5):
    return synth._cfg(n_layers=3, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=157, attn_type=attn, norm_type=norm, act=act,
                      batch=batch, prompt=prompt, steps=4, dtype=dtype)


def _within(gl, lg, what):
    assert np.abs(gl - lg).max() <= FP16_SENSITIVE_REL * np.abs(lg).max(), what


# the tile by size, every tile by itself, and tiles whose K several blocks share (their counters go through graph replays)
TILES = ("", "11", "12", "14", "22", "24", "411", "412", "322", "424")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("max_batch,batch", [(33, 33), (64, 1), (64, 64), (100, 65), (128, 128)])
def test_rows(G, oracle, monkeypatch, shape, max_batch, batch):
    """Steps one by one against the oracle, and the generate loop with and without its captured graph: the same tokens and the
    same bits as those steps.  (A new model per tile: a captured step keeps the tiles it was captured with.)"""
    hidden, heads, kv, ffn, act = shape
    cfg = _cfg(hidden, heads, kv, ffn, synth.RMSNORM, act, batch, "f16")
    w = sensitive(synth.make_weights(cfg, 61, random_bias=True), hidden)
    seqs = synth.make_prompts(cfg, 62)
    orc = oracle.OracleGpt(cfg, w)
    p, lg = orc.step(seqs, use_cache=True)
    want, fed, cur = [lg], [], seqs
    for _ in range(4):
        fed.append(oracle.argmax(p).astype(np.int32))
        cur = np.concatenate([cur, fed[-1][:, None]], 1)
        p, lg = orc.step(cur, use_cache=True)
        want.append(lg)
    for tile in TILES:
        if tile:
            monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
        gpu = G.HipGpt(cfg, w, max_batch=max_batch, max_seq_len=24)
        gpu.prefill(seqs)
        _within(gpu.logits(), want[0], tile)
        for nxt, lg in zip(fed, want[1:]):
            gpu.decode(nxt)
            _within(gpu.logits(), lg, tile)
        assert gpu.seq_len() == seqs.shape[1] + 4
        runs = []
        for graph in (True, False):
            if not graph:
                monkeypatch.setenv("TSHIP_NO_GRAPH", "1")
            gpu.reset()
            gpu.prefill(seqs)
            ids, _ = gpu.generate(4)
            runs.append((ids, gpu.logits()))
        monkeypatch.delenv("TSHIP_NO_GRAPH")
        gpu.reset()
        gpu.prefill(seqs)
        for nxt in runs[0][0]:
            assert np.array_equal(gpu.sample(), nxt), tile
            gpu.decode(nxt)
        for ids, logits in runs:
            assert np.array_equal(ids, runs[0][0]) and np.array_equal(logits, gpu.logits()), tile
        gpu.close()


@pytest.mark.parametrize("dtype,hidden,heads", [("f32", 64, 4), ("f16", 64, 4), ("f16", 128, 2)])
def test_reorder_rows(G, dtype, hidden, heads):
    """Rows of shared prompts, of mixed ones and after a rewind, 1 ... 20 rows: the caches are the gathered ones."""
    cfg = _cfg(hidden, heads, heads, 96, synth.RMSNORM, synth.RELU, 2, dtype, prompt=37)
    w = synth.make_weights(cfg, 71, random_bias=True)
    seqs = synth.make_prompts(cfg, 72)
    gpu = G.HipGpt(cfg, w, max_batch=20, max_seq_len=64)
    rng = np.random.default_rng(73)

    def kv():
        return [gpu.get_kv(l, i) for l in range(3) for i in range(2)]

    def move(src):
        before = kv()
        gpu.reorder_rows(np.array(src, np.int32))
        gpu.decode(rng.integers(4, 157, size=len(src)).astype(np.int32))
        for a, b in zip(before, kv()):
            assert np.array_equal(a[np.array(src)], b[:, :, :a.shape[2]]), src

    gpu.prefill(seqs)
    move([0, 1, 0, 1, 0, 1, 0, 1])                       # two prompts, four hypotheses each
    move([2, 1, 0, 3, 2, 7, 0, 5])                       # inside the prompts: only what was decoded moves
    move([3, 1, 0, 3, 2, 7, 0, 5])                       # a row takes the other prompt's place
    move([7, 0])                                         # fewer rows
    move([1, 0, 1, 1, 0, 0, 1, 0, 1, 1, 0, 0])
    move(list(rng.integers(0, 12, size=16)))
    move(list(rng.integers(0, 16, size=20)))             # more than the in-place kernel takes
    gpu.set_seq_len(20, 20)                              # back into the prompt, then on with different tokens
    gpu.decode(rng.integers(4, 157, size=20).astype(np.int32))
    move(list(rng.integers(0, 20, size=7)))
    gpu.prefill(rng.integers(4, 157, size=(7, 9)).astype(np.int32))
    move([6, 5, 4, 3, 2, 1, 0])
    gpu.close()


def test_rows_left_behind_by_a_move_keep_their_own_prompts(G):
    """A move to fewer rows, a step (profile_decode takes any batch) that takes the rows behind them in again, and a move
    among those: they hold different prompts, so all of a row changes places."""
    cfg = _cfg(64, 4, 4, 96, synth.RMSNORM, synth.RELU, 8, "f32", prompt=70)
    w = synth.make_weights(cfg, 76, random_bias=True)
    gpu = G.HipGpt(cfg, w, max_batch=8, max_seq_len=96)
    gpu.prefill(synth.make_prompts(cfg, 77))
    gpu.reorder_rows(np.array([1, 0, 2, 3], np.int32))
    gpu.profile_decode(np.arange(4, 12, dtype=np.int32))
    before = [gpu.get_kv(l, i) for l in range(3) for i in range(2)]
    src = np.array([0, 1, 2, 3, 5, 4, 7, 6], np.int32)
    gpu.reorder_rows(src)
    for a, b in zip(before, [gpu.get_kv(l, i) for l in range(3) for i in range(2)]):
        assert np.array_equal(a[src], b)
    gpu.close()


@pytest.mark.parametrize("rows", [2, 8, 16])
def test_set_kv_behind_a_move(G, rows):
    """Keys and values handed in right behind a move of whole rows are what the cache holds: the move has ended by then."""
    cfg = _cfg(512, 8, 8, 96, synth.RMSNORM, synth.RELU, rows, "f32")
    w = synth.make_weights(cfg, 74)
    gpu = G.HipGpt(cfg, w, max_batch=rows, max_seq_len=1024)
    gpu.set_seq_len(rows, 1000)
    rng = np.random.default_rng(75)
    new = rng.standard_normal((rows, 8, 1000, 64), dtype=np.float32)
    src = np.roll(np.arange(rows), 1)
    for layer in (0, 2):
        for which in (0, 1):
            gpu.reorder_rows(src)
            gpu.set_kv(layer, which, new)
            assert np.array_equal(gpu.get_kv(layer, which), new), (layer, which)
    gpu.close()


@pytest.mark.parametrize("hidden,heads,kv,ffn,norm,act", SPLIT_SHAPES)
@pytest.mark.parametrize("batch,prompt", [(1, 1), (1, 65), (3, 60), (2, 128)])
def test_prefill_tiles_that_share_k(G, oracle, monkeypatch, hidden, heads, kv, ffn, norm, act, batch, prompt):
    """Two to four blocks per tile (TSHIP_GEMM_TILE from 200 on), k-tile counts 10, 32, 44 and 62.5: ranges of unequal length,
    and counts that leave fewer ranges than asked for; a second prefill finds the counters at zero."""
    cfg = _cfg(hidden, heads, kv, ffn, norm, act, batch, "f16", prompt=prompt)
    w = sensitive(synth.make_weights(cfg, 81, random_bias=True), hidden)
    seqs = synth.make_prompts(cfg, 82)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 8)
    for tile in (211, 311, 411, 212, 414, 222, 322, 424):
        monkeypatch.setenv("TSHIP_GEMM_TILE", str(tile))
        got = []
        for _ in range(2):
            gpu.reset()
            gpu.prefill(seqs)
            got.append(gpu.logits())
        _within(got[0], lg, tile)
        assert np.array_equal(got[0], got[1]), tile
    gpu.close()
