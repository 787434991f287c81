"""MoE prefills of fp16 models whose experts' last rows, less than 256 each, run in a launch of their own, and the router that takes
a row per wavefront: against the oracle."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu
FP16_ABS = 3e-2        # (logits of fp16 models of this size: the bar of the other MoE prefill tests)


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


# 512 rows: fewer than 256 per expert of eight (no whole row tile); as many experts as lanes, some of them without rows
@pytest.mark.parametrize("experts,k,batch,prompt,router_bias", [(64, 2, 3, 210, None), (64, 1, 2, 300, (60.0,) * 5 + (0.0,) * 59), (33, 3, 1, 700, None), (8, 1, 4, 128, None), (4, 2, 5, 520, None), (16, 5, 1, 600, None),
                                                                (4, 2, 2, 256, (60.0, 0.0, 0.0, 0.0)), (4, 2, 3, 200, (-60.0, 0.0, 0.0, 0.0))])
@pytest.mark.parametrize("tile", [11, 12, 14, 22, 24, None])
def test_last_rows_by_themselves(G, oracle, monkeypatch, experts, k, batch, prompt, router_bias, tile):
    """In the third layer of four (the last one computes the last positions only, as a decode step)."""
    cfg = synth.tiny_config(n_layers=4, n_experts=experts, experts_per_token=k, norm_type=synth.LAYERNORM, act=synth.RELU, dtype="f16",
                            batch=batch, prompt=prompt, vocab=300)
    w = synth.make_weights(cfg, 62, random_bias=True)
    if router_bias is not None:
        w["GPTDecoder.MoEFFN_2.m_RouterBias"] = np.asarray(router_bias, np.float32).reshape(1, experts)
    seqs = synth.make_prompts(cfg, 162)
    if tile is not None:
        monkeypatch.setenv("TSHIP_MOE_REST", str(tile))
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 10)
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    gpu.prefill(seqs)
    got = gpu.logits()
    kernels = gpu.profile_symbols()
    assert any("moe_lists_big_kernel" in s for s in kernels) and not any("moe_gather_kernel" in s for s in kernels)      # one launch for all experts
    if tile is not None:      # (its last template argument: the last rows of several problems)
        assert sum("mid_gemm_f16_kernel" in s and ", %d, %d, true>" % (tile // 10, tile % 10) in s for s in kernels) == 2
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    assert np.abs(got - lg).max() <= FP16_ABS
    gpu.close()


# hidden sizes that fill no row of lanes, four and eight column groups per lane, expert counts around eight; more rows than wavefronts;
# and matrices that leave no room in LDS (fast: a block per row instead)
@pytest.mark.parametrize("hidden,heads,kv,experts,k,batch,prompt,fast",
                         [(48, 3, 1, 2, 1, 1, 3, True), (64, 4, 2, 9, 4, 3, 90, True), (528, 33, 11, 8, 2, 2, 40, True), (64, 4, 4, 64, 4, 1, 60, True), (64, 4, 2, 8, 2, 9, 500, True),
                          (272, 17, 17, 16, 2, 2, 300, True), (1056, 33, 11, 8, 3, 1, 17, True), (1040, 65, 13, 7, 4, 2, 30, True), (2048, 32, 8, 3, 2, 1, 40, True),
                          (1056, 33, 11, 12, 3, 1, 17, False), (2080, 65, 13, 7, 2, 1, 9, False)])
def test_router_of_many_rows(G, oracle, monkeypatch, hidden, heads, kv, experts, k, batch, prompt, fast):
    cfg = synth.tiny_config(n_layers=3, hidden=hidden, n_heads=heads, n_kv_heads=kv, n_experts=experts, experts_per_token=k, norm_type=synth.LAYERNORM,
                            act=synth.RELU, dtype="f16", batch=batch, prompt=prompt, vocab=100)
    w = synth.make_weights(cfg, 63, random_bias=True)
    monkeypatch.setenv("TSHIP_MOE_ROUTER_ROWS", "0")
    monkeypatch.setenv("TSHIP_ALL_ROWS", "1")
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    seqs = synth.make_prompts(cfg, 163)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 10)
    gpu.prefill(seqs)
    routers = [s for s in gpu.profile_symbols() if "moe_router" in s]
    assert routers and all(("moe_router_rows_kernel<%d>" % (4 if hidden <= 1024 else 8) in s) == fast for s in routers)
    orc = oracle.OracleGpt(cfg, w)
    _, lg = orc.step(seqs, use_cache=True)
    assert np.abs(gpu.logits() - lg).max() <= FP16_ABS
    ti, tv, pr = gpu.moe_routing(2)
    op = orc.moe_trace(0)[2].reshape(batch, prompt, experts)[:, -1]
    assert np.abs(pr - op).max() <= 5e-3                # fp16 activations in front of the router
    order = np.argsort(-pr, axis=1, kind="stable")[:, :k]
    assert np.array_equal(tv, np.take_along_axis(pr, ti.astype(int), 1)) and np.array_equal(tv, np.take_along_axis(pr, order, 1))
    gpu.close()
