"""The QKV projection of an fp16 prefill writing the fragment-major cache in pieces, against the kernel that does it behind the
projection (TSHIP_NO_KV_FUSE), bit for bit."""
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


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,prompt,context", [(1, 1, 0), (1, 31, 0), (2, 33, 0), (3, 65, 20), (2, 40, 32), (5, 128, 0), (1, 700, 0), (9, 5, 7)])
def test_cache_in_pieces(G, monkeypatch, shape, batch, prompt, context):
    """Prompts that end inside and at 32-position chunks, shorter than a chunk's rest, behind a context; every kind of tile, whole and
    partly beyond the matrix; twice over a cache that a longer prompt has filled, and two steps behind it."""
    hidden, heads, kv, norm = SHAPES[shape]
    cfg = synth._cfg(n_layers=2, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=192, vocab=157, attn_type=synth.GQA, norm_type=norm, act=synth.RELU,
                     batch=batch, prompt=context + prompt, steps=2, dtype="f16")
    w = synth.make_weights(cfg, 111, random_bias=True)
    seqs = synth.make_prompts(cfg, 112)
    longer = np.random.default_rng(113).integers(4, 157, size=(batch, context + prompt + 40)).astype(np.int32)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=context + prompt + 48)
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    for tile in (None, "0", "11", "14", "222", "24", "42", "43", "45"):
        if tile:
            monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
        got = []
        for separate in (False, True):
            if separate:
                monkeypatch.setenv("TSHIP_NO_KV_FUSE", "1")
            gpu.reset()
            gpu.prefill(longer)
            gpu.reset()
            if context:
                gpu.prefill(seqs[:, :context])
            gpu.prefill(seqs[:, context:])
            assert any("kv_write" in s for s in gpu.profile_symbols()) == separate, tile
            out = [gpu.logits()] + [gpu.get_kv(l, i) for l in range(2) for i in range(2)]
            for _ in range(2):
                gpu.decode((np.arange(batch) + 5).astype(np.int32))
                out.append(gpu.logits())
            got.append(out)
        monkeypatch.delenv("TSHIP_NO_KV_FUSE")
        for a, b in zip(*got):
            assert np.array_equal(a, b), tile
    gpu.close()
