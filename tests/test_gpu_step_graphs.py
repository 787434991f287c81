"""Token loops long enough for the captured graph of eight steps, which a call of 16 steps or more makes behind its sixteenth, a shorter one
behind its last once 64 steps have run: the tokens and logits of steps launched one by one."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


@pytest.mark.parametrize("dtype,norm,batch,experts", [("f16", synth.RMSNORM, 3, 1), ("f16", synth.LAYERNORM, 2, 1), ("f16", synth.RMSNORM, 40, 1), ("f32", synth.RMSNORM, 2, 1),
                                                      ("f16", synth.LAYERNORM, 4, 4)])
@pytest.mark.parametrize("sampled", [False, True])
def test_loops_of_many_steps(G, monkeypatch, dtype, norm, batch, experts, sampled):
    """Loops that make the long graph and run it at once (64, 47, 24), make it and leave it to a later one (16 to 23; the last of them at the
    cache's end), are too short for it (15, the first calls of 8), and find it there, below, at and between multiples of eight steps; a rewind, single
    steps, a loop that looks for an end token and blocked tokens (which drop the graphs) between them; the same where the long graph
    cannot be made.  (Models with experts make none.)"""
    cfg = synth.tiny_config(n_layers=3, dtype=dtype, norm_type=norm, n_experts=experts, experts_per_token=min(2, experts), batch=batch, prompt=8, vocab=300,
                             act=synth.RELU if experts > 1 else synth.SWIGLU)
    w = synth.make_weights(cfg, 101, random_bias=True)
    seqs = synth.make_prompts(cfg, 102)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=160)
    if sampled:
        gpu.set_repeat_penalty(2.0)

    def loop(n, until=None):
        args = (G.TOPP, 0.9, 1.0, synth.make_uniforms(103 + n, batch, n)) if sampled else (G.GREEDY,)
        ids = (gpu.generate_until(n, until, *args) if until is not None else gpu.generate(n, *args))[0]
        return np.array(ids), gpu.logits()

    def run():
        gpu.set_blocked_tokens([])
        gpu.reset()
        gpu.prefill(seqs)
        out = [loop(64), loop(7), loop(8), loop(29)]
        gpu.set_seq_len(batch, 40)
        gpu.decode((np.arange(batch) + 4).astype(np.int32))
        out += [loop(19), loop(9, until=2), loop(16)]
        gpu.set_blocked_tokens([5, 6, 7])
        out += [loop(31), loop(20)]

        def again(at, *lengths):
            gpu.set_seq_len(batch, at)
            gpu.decode((np.arange(batch) + 4).astype(np.int32))
            return [loop(n) for n in lengths]

        for lengths in ((32, 33, 10), (47, 9, 10), (24, 8), (15, 16, 23), (8,) * 10):
            gpu.set_blocked_tokens([])
            out += again(40, *lengths)
            gpu.set_blocked_tokens([5])
        out += again(160 - 17, 16) + again(40, 24)
        return out

    first, second = run(), run()
    monkeypatch.setenv("TSHIP_FAIL_STEPS_GRAPH", "1")
    gpu.set_blocked_tokens([5])
    without = run()
    monkeypatch.setenv("TSHIP_NO_GRAPH", "1")
    want = run()
    for got in (first, second, without):
        for (a, la), (b, lb) in zip(got, want):
            assert np.array_equal(a, b) and np.array_equal(la, lb)
    gpu.close()
