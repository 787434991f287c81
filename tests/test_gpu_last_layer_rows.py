"""Prefills compute the last layer behind its keys and values for the last positions only: against the oracle, and against the
same layer with all rows."""
import numpy as np
import pytest

from parity_util import FP16_SENSITIVE_REL, sensitive
from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


# hidden, heads, kv heads, ffn, norm, activation, dtype, layers, experts: head sizes 16 to 128, deferred and stored norms, a last layer with experts
SHAPES = {
    "f16_rms_d16": (160, 10, 5, 200, synth.RMSNORM, synth.SWIGLU, "f16", 2, 1),
    "f16_rms_d64": (512, 8, 2, 704, synth.RMSNORM, synth.SWIGLU_SILU, "f16", 1, 1),
    "f16_rms_d128": (512, 4, 2, 704, synth.RMSNORM, synth.SWIGLU, "f16", 2, 1),
    "f16_ln_d64": (192, 3, 3, 104, synth.LAYERNORM, synth.RELU, "f16", 2, 1),
    "f32_d64": (256, 4, 4, 300, synth.LAYERNORM, synth.RELU, "f32", 2, 1),
    "f32_d16_gated": (48, 3, 1, 104, synth.RMSNORM, synth.SWIGLU, "f32", 1, 1),
    "f16_moe": (128, 2, 1, 256, synth.LAYERNORM, synth.RELU, "f16", 4, 8),
    "f32_moe": (64, 4, 2, 128, synth.LAYERNORM, synth.RELU, "f32", 3, 4),
}


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,prompt,context,padded", [(1, 2, 0, False), (1, 33, 0, False), (3, 65, 20, False), (2, 300, 32, False), (33, 17, 0, False), (5, 128, 0, True)])
def test_last_positions(G, oracle, monkeypatch, shape, batch, prompt, context, padded):
    """Two positions, prompts that end inside and at blocks of queries, behind a context, more than 32 rows, padded: logits, hidden
    state and the routing of the last positions, and two steps behind them, which read the cache.  The front layers and the last one's
    keys and values are computed alike with all rows (TSHIP_ALL_ROWS), so the cache and those steps are the same bits."""
    hidden, heads, kv, ffn, norm, act, dtype, layers, experts = SHAPES[shape]
    total = context + prompt
    cfg = synth._cfg(n_layers=layers, hidden=hidden, n_heads=heads, n_kv_heads=kv, ffn_dim=ffn, vocab=157, attn_type=synth.GQA, norm_type=norm, act=act,
                     n_experts=experts, experts_per_token=min(2, experts), batch=batch, prompt=total, steps=2, dtype=dtype)
    w = synth.make_weights(cfg, 95, random_bias=True)
    if experts == 1:
        w = sensitive(w, hidden)
    seqs = synth.make_prompts(cfg, 96)
    lens = None
    if padded:
        lens = np.array([prompt, 1, prompt // 2, prompt - 1, 33][:batch], np.int32)
        seqs, lens = G.HipGpt.pad_sentences([row[:n] for row, n in zip(seqs, lens)], pad_id=0)
    orc = oracle.OracleGpt(cfg, w)
    if padded:
        _, lg = orc.step(seqs, use_cache=True, lens=lens.astype(np.float32))
    else:
        _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=total + 8)

    def run():
        gpu.reset()
        if context:
            gpu.prefill(seqs[:, :context])
        gpu.prefill(seqs[:, context:], lens)
        behind = [gpu.logits(), gpu.hidden()] + (list(gpu.moe_routing(layers - 1)) if experts > 1 else [])
        exact = [gpu.get_kv(l, i) for l in range(layers) for i in range(2)]
        for _ in range(2):
            gpu.decode((np.arange(batch) + 5).astype(np.int32))
            exact.append(gpu.logits())
        return behind, exact

    last, exact = run()
    monkeypatch.setenv("TSHIP_ALL_ROWS", "1")
    rows, exact_rows = run()
    for a, b in zip(exact, exact_rows):
        assert np.array_equal(a, b)
    scale = np.abs(lg).max()
    bar = 1e-4 * scale if dtype == "f32" else FP16_SENSITIVE_REL * scale if experts == 1 else 3e-2      # (the bars of the other prefill tests)
    assert np.abs(last[0] - lg).max() <= bar and np.abs(last[0] - rows[0]).max() <= bar
    # fp32 sums in another order; fp16: of the products of the feed-forward, rounded to 2^-11 of themselves, a few round the other way
    assert np.abs(last[1] - rows[1]).max() <= (1e-5 if dtype == "f32" else 2e-3) * np.abs(rows[1]).max()
    if experts > 1:
        top, value, probs = last[2:]
        want = orc.moe_trace(layers - 3)[2].reshape(batch, total, experts)[:, -1]
        assert np.abs(probs - want).max() <= (1e-5 if dtype == "f32" else 5e-3)      # (fp16 activations in front of the router)
        order = np.argsort(-probs, axis=1, kind="stable")[:, :2]
        assert np.array_equal(value, np.take_along_axis(probs, order, 1)) and np.array_equal(value, np.take_along_axis(probs, top.astype(int), 1))
        if dtype == "f32":
            assert np.array_equal(top, np.argsort(-want, axis=1, kind="stable")[:, :2])
        assert np.array_equal(top, rows[2]) and np.abs(probs - rows[4]).max() <= 1e-4      # (the router's input: fp32 sums in another order)
    gpu.close()


@pytest.mark.parametrize("switch", [{}, {"TSHIP_MOE_REST": "12"}, {"TSHIP_MOE_ROUTER_ROWS": "100"}, {"TSHIP_GEMM_TILE": "0"}])
def test_what_is_recorded_is_what_runs(G, monkeypatch, switch):
    """The kernels recorded of a prefill, with a tile or a router forced or not, hold those of a last layer that computes the last positions: a
    decode step's router behind the one of all rows.  Recording them changes no bit of the logits."""
    cfg = synth.tiny_config(n_layers=4, n_experts=4, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU, dtype="f16", batch=3, prompt=400, vocab=300)
    seqs = synth.make_prompts(cfg, 99)
    gpu = G.HipGpt(cfg, synth.make_weights(cfg, 98, random_bias=True), max_batch=3, max_seq_len=404)
    for name, value in switch.items():
        monkeypatch.setenv(name, value)
    got = []
    for record in (False, True):
        if record:
            monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
        gpu.reset()
        gpu.prefill(seqs)
        got.append(gpu.logits())
    routers = [s for s in gpu.profile_symbols() if "moe_router" in s]
    assert len(routers) == 2 and "moe_router_rows_kernel" in routers[0] and "moe_router_fast_kernel" in routers[1]
    assert np.array_equal(*got)
    monkeypatch.setenv("TSHIP_ALL_ROWS", "1")
    gpu.reset()
    gpu.prefill(seqs)
    assert sum("moe_router_rows_kernel" in s for s in gpu.profile_symbols()) == 2
    gpu.close()


@pytest.mark.parametrize("experts,k,batch,prompt,router_bias", [(4, 1, 5, 520, None), (16, 4, 2, 300, None), (4, 2, 3, 200, (-60.0, 0.0, 0.0, 0.0)), (4, 2, 3, 200, (60.0, 0.0, 0.0, 0.0))])
def test_a_layer_of_experts_in_front_of_the_last(G, oracle, monkeypatch, experts, k, batch, prompt, router_bias):
    """One launch for all experts against one per expert, bit for bit, where a layer that computes all rows has them."""
    cfg = synth.tiny_config(n_layers=4, n_experts=experts, experts_per_token=k, norm_type=synth.LAYERNORM, act=synth.RELU, dtype="f16",
                            batch=batch, prompt=prompt, vocab=300)
    w = dict(synth.make_weights(cfg, 97, random_bias=True))
    if router_bias is not None:
        w["GPTDecoder.MoEFFN_2.m_RouterBias"] = np.asarray(router_bias, np.float32).reshape(1, experts)
    seqs = synth.make_prompts(cfg, 98)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 10)
    gpu.prefill(seqs)
    one = [gpu.logits(), gpu.get_kv(3, 0), gpu.get_kv(3, 1)]
    monkeypatch.setenv("TSHIP_NO_MOE_BATCH", "1")
    gpu.reset()
    gpu.prefill(seqs)
    for a, b in zip(one, [gpu.logits(), gpu.get_kv(3, 0), gpu.get_kv(3, 1)]):
        assert np.array_equal(a, b)
    assert np.abs(one[0] - lg).max() <= 3e-2
    gpu.close()
