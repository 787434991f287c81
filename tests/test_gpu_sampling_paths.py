"""Token choice from the logits: top-p rows finished from their largest candidates and rows that need the sort, in one batch; up to
eight greedy beam picks at once and more than eight; the greedy scan at odd vocabulary sizes.  The oracle gets the softmax of the
device's own logits, so that both sides choose from the same distribution; all sampled comparisons are of whole numbers."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu
HEAD, BIAS = "FeedForward_Decoder_0.m_Whd", "FeedForward_Decoder_0.m_Bd"


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _model(G, vocab, batch, dtype, bias, head=1.0, hidden=64):
    cfg = synth.tiny_config(vocab=vocab, batch=batch, prompt=6, dtype=dtype, hidden=hidden, n_heads=hidden // 16, n_kv_heads=hidden // 32)
    w = synth.make_weights(cfg, 7, random_bias=True)
    w[HEAD] = (w[HEAD] * np.float32(head)).astype(np.float32)
    w[BIAS] = np.asarray(bias, np.float32).reshape(w[BIAS].shape)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=48)
    seqs = synth.make_prompts(cfg, 8) if vocab > 4 else np.zeros((batch, 6), np.int32)
    gpu.prefill(seqs)
    return gpu, seqs


def _probs(oracle, gpu, temperature=1.0):
    return oracle.softmax((gpu.logits() / np.float32(temperature)).astype(np.float32))


# bias spread 3: a few hundred candidates at most reach 2^-9; 0: none does in a large vocabulary; top_p None: between the masses
# that the rows' large candidates have, so that some rows are finished from them and the others sorted
@pytest.mark.parametrize("dtype,hidden", [("f32", 64), ("f16", 256)])
@pytest.mark.parametrize("vocab,spread,top_p", [(61, 1.0, 0.9), (513, 0.0, 0.9), (1025, 3.0, None), (4099, 3.0, None), (4099, 4.0, 0.5), (4099, 0.0, 0.3)])
@pytest.mark.parametrize("penalty,block,temperature", [(0.0, False, 1.0), (2.0, True, 0.8)])
def test_top_p(G, oracle, dtype, hidden, vocab, spread, top_p, penalty, block, temperature):
    batch, steps = 9, 4
    gpu, seqs = _model(G, vocab, batch, dtype, np.random.default_rng(3).normal(0.0, spread, vocab), head=8.0, hidden=hidden)
    blocked = [0, 5, vocab - 1] if block else []
    u = synth.make_uniforms(9, batch, steps)

    def start():
        gpu.reset()
        if penalty:
            gpu.set_repeat_penalty(penalty)
        gpu.prefill(seqs)

    if block:
        gpu.set_blocked_tokens(blocked)
    start()
    p = _probs(oracle, gpu, temperature)
    if top_p is None:
        mass = np.sort(np.where(p >= 2.0 ** -9, p, 0).sum(1))
        top_p = float(mass[4] + mass[5]) / 2
        assert mass[0] < top_p < mass[-1]
    cur, want = seqs, []
    for s in range(steps):
        p = _probs(oracle, gpu, temperature)
        p[:, blocked] -= 1.0
        want.append(oracle.toppsample(p, top_p, penalty, cur if penalty else None, u[s]).astype(np.int32))
        assert np.array_equal(gpu.sample(mode=G.TOPP, top_p=top_p, temperature=temperature, uniforms=u[s]), want[-1])
        cur = np.concatenate([cur, want[-1][:, None]], 1)
        gpu.decode(want[-1])
    start()
    ids, _ = gpu.generate(steps, mode=G.TOPP, top_p=top_p, temperature=temperature, uniforms=u)      # the replayed step: every replay chooses anew
    assert np.array_equal(ids, np.stack(want))
    gpu.close()


# whole-number logits: ties everywhere; "cliff": all but six tokens have probability zero, so that later picks are of zeros and of
# tokens picked before
@pytest.mark.parametrize("vocab", [9, 61, 1023, 1025, 5003])
@pytest.mark.parametrize("kind", ["ties", "cliff", "rows"])
@pytest.mark.parametrize("block", [False, True])
def test_greedy_beam_picks(G, oracle, vocab, kind, block):
    rng = np.random.default_rng(vocab)
    bias = rng.integers(0, 4, vocab).astype(np.float32)
    if kind == "cliff":
        bias = np.full(vocab, -1000.0, np.float32)
        bias[rng.permutation(vocab)[:6]] = 1.0
    gpu, _ = _model(G, vocab, 3, "f32", bias, head=8.0 if kind == "rows" else 0.0)
    p = _probs(oracle, gpu)
    if block:
        blocked = [int(np.argmax(p[0])), vocab - 1]
        gpu.set_blocked_tokens(blocked)
        p[:, blocked] -= 1.0
    assert np.array_equal(gpu.sample(), oracle.argmax(p).astype(np.int32))
    n_all = min(9, vocab - 2)
    ids9, logp9 = gpu.beam_pick(n_all)
    for n in (1, 2, 5, min(8, n_all)):
        ids, logp = gpu.beam_pick(n)
        want, wlogp = oracle.beam_picks(p, n)
        assert np.array_equal(ids, want) and np.array_equal(ids, ids9[:n])
        assert np.allclose(logp, wlogp, rtol=1e-5, atol=1e-5) and np.allclose(logp, logp9[:n], rtol=1e-5, atol=1e-5)
    gpu.close()


@pytest.mark.parametrize("vocab", [1, 3, 4097, 32769])
def test_greedy_scan_finds_every_position(G, oracle, vocab):
    """The largest logit at the ends of the row and of the 16-byte pieces, with a tie behind it."""
    for at in sorted({0, vocab // 2, max(vocab - 2, 0), vocab - 1}):
        bias = np.zeros(vocab, np.float32)
        bias[at:] = 2.0
        gpu, _ = _model(G, vocab, 2, "f32", bias, head=0.0)
        assert np.array_equal(gpu.sample(), [at, at])
        gpu.close()
