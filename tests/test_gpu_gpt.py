"""Parity of the fused GPTDecoder path (TSHip_Gpt*) with the CPU oracle on identical seeded weights and inputs.

Bars (from the benchmark contract): fp32 logits max relative error <= 1e-4 and identical greedy tokens; fp16
logits max absolute error <= 3e-2 and >= 99 % per-step top-1 agreement under teacher forcing (the fp16 oracle is
the fp32 CPU path on fp16-rounded weights: the reference's CPU backend is fp32 only); KV-cache indexing, token
gathers and MoE routing bit-exact; top-p driven by a shared seeded uniform stream."""
import json
import os

import numpy as np
import pytest

from parity_util import top1_agreement
from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")

FP32_REL = 1e-4
FP16_ABS = 3e-2


@pytest.fixture(scope="module")
def G():
    from seq2seqsharp_amd import gpt
    return gpt


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _teacher_forced(G, oracle, cfg, seed, steps, **kw):
    """Prefill + `steps` decode steps feeding both sides the oracle's greedy tokens; yields per-step logits."""
    w = synth.make_weights(cfg, seed, random_bias=True)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=cfg["batch"], max_seq_len=cfg["prompt"] + steps + 2, **kw)
    seqs = synth.make_prompts(cfg, seed + 100)
    p, lg = orc.step(seqs, use_cache=True)
    gpu.prefill(seqs)
    out = [(lg, gpu.logits())]
    cur = seqs
    for _ in range(steps):
        nxt = oracle.argmax(p).astype(np.int32)
        cur = np.concatenate([cur, nxt[:, None]], 1)
        p, lg = orc.step(cur, use_cache=True)
        gpu.decode(nxt)
        out.append((lg, gpu.logits()))
    return orc, gpu, out, cur


TINY = {
    "gqa_rms_gate": dict(),
    "mha_ln_relu": dict(attn_type=synth.MHA, n_kv_heads=4, norm_type=synth.LAYERNORM, act=synth.RELU),
    "gqa_rms_silu": dict(act=synth.SILU),
    "gqa_rms_gate_silu": dict(act=synth.SWIGLU_SILU),
    "gqa_leaky_d32_g4": dict(hidden=128, n_heads=4, n_kv_heads=1, act=synth.LEAKYRELU, batch=3, prompt=11, vocab=131),
    "mha_d64": dict(hidden=128, n_heads=2, n_kv_heads=2, attn_type=synth.MHA, batch=1, prompt=5),
    "odd_sizes": dict(hidden=96, n_heads=6, n_kv_heads=3, ffn_dim=200, vocab=1000, batch=5, prompt=13),
}


@pytest.mark.parametrize("name", sorted(TINY))
def test_fp32_logits_and_tokens(G, oracle, name):
    cfg = synth.tiny_config(**TINY[name])
    orc, gpu, out, _ = _teacher_forced(G, oracle, cfg, 3, 6)
    for lg, gl in out:
        assert _rel(gl, lg) <= FP32_REL
        assert np.array_equal(gl.argmax(1), lg.argmax(1))
    gpu.close()


@pytest.mark.parametrize("name", sorted(TINY))
def test_fp16_logits_and_top1(G, oracle, name):
    cfg = synth.tiny_config(dtype="f16", **TINY[name])
    orc, gpu, out, _ = _teacher_forced(G, oracle, cfg, 4, 6)
    agree = []
    for lg, gl in out:
        assert np.abs(gl - lg).max() <= FP16_ABS
        agree.append((gl.argmax(1) == lg.argmax(1)).mean())
    assert np.mean(agree) >= 0.99
    gpu.close()


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_kv_cache_rows_and_indexing(G, oracle, dtype):
    """Every cached row lands at [batch, kv_head, position]; keys are stored after RoPE.  The reference's cache is
    [B*H, d, T] (keys, transposed, heads expanded) and [B*H, T, d] (values): compare through that mapping."""
    cfg = synth.tiny_config(dtype=dtype, batch=3, prompt=7)
    orc, gpu, _, _ = _teacher_forced(G, oracle, cfg, 5, 4)
    H, Gk = cfg["n_heads"], cfg["n_kv_heads"]
    d, B = cfg["hidden"] // H, cfg["batch"]
    T = gpu.seq_len()
    assert T == cfg["prompt"] + 4 == orc.cache_len()
    tol = 1e-5 if dtype == "f32" else 2e-3
    for layer in range(cfg["n_layers"]):
        ko = orc.get_cache(layer, 0).reshape(B, H, d, T)
        vo = orc.get_cache(layer, 1).reshape(B, H, T, d)
        kg, vg = gpu.get_kv(layer, 0), gpu.get_kv(layer, 1)
        for h in range(H):                                   # query head h reads kv head h // (H / Gk)
            assert np.abs(kg[:, h // (H // Gk)] - ko[:, h].transpose(0, 2, 1)).max() <= tol
            assert np.abs(vg[:, h // (H // Gk)] - vo[:, h]).max() <= tol
    gpu.close()


def test_golden_vectors(G):
    """The committed oracle vectors (tests/golden) without the oracle in the loop."""
    meta = json.load(open(os.path.join(GOLD, "tiny_models.json")))
    data = np.load(os.path.join(GOLD, "tiny_models.npz"))
    for case in meta["cases"]:
        cfg = case["cfg"]
        w = synth.make_weights(cfg, case["weight_seed"], random_bias=True)
        gpu = G.HipGpt(cfg, w, max_batch=cfg["batch"], max_seq_len=cfg["prompt"] + case["steps"] + 2)
        toks, logits = data[case["name"] + "_tokens"], data[case["name"] + "_logits"]
        P = cfg["prompt"]
        gpu.prefill(toks[:, :P])
        f16 = cfg["dtype"] == "f16"
        for s in range(case["steps"] + 1):
            gl = gpu.logits()
            if f16:
                assert np.abs(gl - logits[s]).max() <= FP16_ABS
            else:
                assert _rel(gl, logits[s]) <= FP32_REL
                assert np.array_equal(gpu.sample(), toks[:, P + s])
            if s < case["steps"]:
                gpu.decode(toks[:, P + s])
        gpu.close()


def test_generate_matches_stepwise_and_is_deterministic(G):
    cfg = synth.tiny_config(dtype="f16", batch=4, prompt=9)
    w = synth.make_weights(cfg, 7, random_bias=True)
    seqs = synth.make_prompts(cfg, 8)
    gpu = G.HipGpt(cfg, w, max_batch=4, max_seq_len=64)
    gpu.prefill(seqs)
    ids, ms = gpu.generate(12)
    assert ids.shape == (12, 4) and ms > 0 and gpu.seq_len() == 9 + 12
    gpu.reset()
    gpu.prefill(seqs)
    step = []
    for _ in range(12):
        t = gpu.sample()
        step.append(t)
        gpu.decode(t)
    assert np.array_equal(ids, np.stack(step))
    gpu.reset()
    gpu.prefill(seqs)
    ids2, _ = gpu.generate(12)
    assert np.array_equal(ids, ids2)                       # split-K partials are summed in a fixed order
    # the captured step graph replayed in pieces, with eager steps and synchronisations in between
    gpu.reset()
    gpu.prefill(seqs)
    a, _ = gpu.generate(5)
    t = gpu.sample()
    gpu.decode(t)
    b, _ = gpu.generate(3)
    t2 = gpu.sample()
    gpu.decode(t2)
    c, _ = gpu.generate(2)
    assert np.array_equal(np.concatenate([a, t[None], b, t2[None], c]), ids)
    u = synth.make_uniforms(3, 4, 6)
    gpu.reset()
    gpu.prefill(seqs)
    p1, _ = gpu.generate(6, mode=G.TOPP, top_p=0.8, uniforms=u)
    gpu.reset()
    gpu.prefill(seqs)
    p2 = []
    for s in range(6):
        t = gpu.sample(mode=G.TOPP, top_p=0.8, uniforms=u[s])
        p2.append(t)
        gpu.decode(t)
    assert np.array_equal(p1, np.stack(p2))
    gpu.close()


@pytest.mark.parametrize("batch", [4, 8])
def test_decode_equals_prefill_recompute(G, batch):
    """(batch 8: 768 and 800 prompt rows, half of them with batch 4: prefill GEMM tiles of different heights.)
    Size-independent property at the real head shape (GQA 32/8 heads of 64): prefill(P) + decode(tokens) must give
    the logits of prefill(P + n).  It exercises cache positions, the RoPE offset and the decode GEMM against the
    prefill GEMM on a model wide enough to use full MFMA tiles."""
    cfg = dict(synth.CONFIGS["cfg2_1b_gqa_f16"], n_layers=2, vocab=4096, batch=batch, prompt=96)
    w = synth.make_weights(cfg, 9)
    seqs = synth.make_prompts(cfg, 10, length=100)
    a = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=128)
    a.prefill(seqs[:, :96])
    for t in range(96, 100):
        a.decode(seqs[:, t])
    la = a.logits()
    b = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=128)
    b.prefill(seqs)
    lb = b.logits()
    assert np.abs(la - lb).max() <= 2e-2
    assert (la.argmax(1) == lb.argmax(1)).all()
    ka, kb = a.get_kv(1, 0), b.get_kv(1, 0)
    assert np.abs(ka - kb).max() <= 2e-2
    a.close()
    b.close()


def test_full_size_cfg2_properties(G):
    """The benchmark configuration at its real size (16 layers, batch 32, prompt 1024), where the oracle would need
    minutes: prefill(P) + two decode steps must reproduce prefill(P + 2); a KV cache read back and restored into a
    second model agrees; generate() equals step-by-step greedy decoding on the same model, bit for bit."""
    cfg = dict(synth.CONFIGS["cfg2_1b_gqa_f16"])
    B, Tp = cfg["batch"], cfg["prompt"]
    w = synth.make_weights(cfg, 0)
    seqs = synth.make_prompts(cfg, 1, length=Tp + 2)
    a = G.HipGpt(cfg, w, max_batch=B, max_seq_len=Tp + 16)
    a.prefill(seqs[:, :Tp])
    a.decode(seqs[:, Tp])
    a.decode(seqs[:, Tp + 1])
    la = a.logits()
    b = G.HipGpt(cfg, w, max_batch=B, max_seq_len=Tp + 16)
    b.prefill(seqs)
    lb = b.logits()
    assert np.abs(la - lb).max() <= FP16_ABS
    assert (la.argmax(1) == lb.argmax(1)).mean() >= 0.99
    # cache round trip through the host layout [batch, kv_head, len, head_dim]
    for layer in (0, cfg["n_layers"] - 1):
        for which in (0, 1):
            kv = a.get_kv(layer, which)
            assert kv.shape == (B, cfg["n_kv_heads"], Tp + 2, cfg["hidden"] // cfg["n_heads"])
            assert np.abs(kv - b.get_kv(layer, which)).max() <= 2e-2
    g1, _ = a.generate(4)
    # rewind the same model to the end of the prompt and walk the same four steps one call at a time
    a.set_seq_len(B, Tp + 1)
    a.decode(seqs[:, Tp + 1])
    assert np.array_equal(a.logits(), la)
    steps = []
    for _ in range(4):
        nxt = a.sample()
        steps.append(nxt)
        a.decode(nxt)
    assert np.array_equal(g1, np.stack(steps))
    a.close()
    b.close()


@pytest.mark.parametrize("tile", ["by_size", "0"])
@pytest.mark.parametrize("name", ["odd_sizes", "gqa_leaky_d32_g4", "mha_ln_relu"])
def test_fp16_long_prompt_prefill_against_oracle(G, oracle, monkeypatch, name, tile):
    """655 prompt rows: the prefill projections with the tile picked by size, and with 256 x 256 tiles (ragged row, column
    and k tiles with these sizes).  Logits of the last position and the whole KV cache of the last layer against the oracle."""
    if tile != "by_size":
        monkeypatch.setenv("TSHIP_GEMM_TILE", tile)
    cfg = synth.tiny_config(dtype="f16", **dict(TINY[name], batch=5, prompt=131))
    w = synth.make_weights(cfg, 21, random_bias=True)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=5, max_seq_len=140)
    seqs = synth.make_prompts(cfg, 22)
    _, lg = orc.step(seqs, use_cache=True)
    gpu.prefill(seqs)
    gl = gpu.logits()
    assert np.abs(gl - lg).max() <= FP16_ABS
    assert top1_agreement(gl, lg)[0] >= 0.99          # (these tiny models have near-equal leading logits: ties are not misses)
    H, Gk = cfg["n_heads"], cfg["n_kv_heads"]
    d = cfg["hidden"] // H
    last = cfg["n_layers"] - 1
    kc, vc = orc.get_cache(last, 0), orc.get_cache(last, 1)
    ko = kc.reshape(5, H, d, 131)[:, ::H // Gk].transpose(0, 1, 3, 2)       # reference keeps K as [B*H, d, T]
    vo = vc.reshape(5, H, 131, d)[:, ::H // Gk]
    assert np.abs(gpu.get_kv(last, 0) - ko).max() <= 2e-2
    assert np.abs(gpu.get_kv(last, 1) - vo).max() <= 2e-2
    gpu.close()


def test_topp_stream_matches_oracle(G, oracle):
    """Both sides consume the same pre-generated uniform stream, one draw per row per step (ComputeGraphTensor.cs:2379).
    fp32 model: probabilities agree to ~1e-7, so the chosen tokens agree unless a draw lands within that distance of a
    bucket boundary; the seeds below have no such draw."""
    cfg = synth.tiny_config(vocab=500, batch=4)
    w = synth.make_weights(cfg, 21, random_bias=True)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=4, max_seq_len=64)
    seqs = synth.make_prompts(cfg, 22)
    u = synth.make_uniforms(23, 4, 10)
    gpu.prefill(seqs)
    ids, _ = gpu.generate(10, mode=G.TOPP, top_p=0.9, temperature=1.0, uniforms=u)
    cur = seqs
    for s in range(10):
        p, _ = orc.step(cur, use_cache=True, sampling=True)
        nxt = oracle.toppsample(p, 0.9, 0.0, None, u[s]).astype(np.int32)
        assert np.array_equal(ids[s], nxt)
        cur = np.concatenate([cur, nxt[:, None]], 1)
    # temperature other than 1 divides the logits first (Decoder.cs:720-723)
    gpu.reset()
    gpu.prefill(seqs)
    orc.reset()
    p, _ = orc.step(seqs, use_cache=True, temperature=0.7, sampling=True)
    got = gpu.sample(mode=G.TOPP, top_p=0.5, temperature=0.7, uniforms=u[0])
    assert np.array_equal(got, oracle.toppsample(p, 0.5, 0.0, None, u[0]).astype(np.int32))
    gpu.close()


@pytest.mark.parametrize("moe", [False, True])
def test_topp_repeat_penalty_matches_oracle(G, oracle, moe):
    """Decoder.cs:761 hands TopPSample the sequences so far (prompt + generated) and DecodingOptions.RepeatPenalty
    (default 2): the device keeps the last position of every token and decays on the fly.  Graph loop, the stepwise
    calls and the token-by-token prompt path of MoE models must all see the same history."""
    from seq2seqsharp_amd._lib import TSHipError
    kw = dict(n_layers=3, n_experts=4, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU) if moe else {}
    cfg = synth.tiny_config(vocab=300, batch=4, **kw)
    w = synth.make_weights(cfg, 31, random_bias=True)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=4, max_seq_len=64)
    seqs = synth.make_prompts(cfg, 32)
    seqs[:, 3] = seqs[:, 1]                                             # repeats inside the prompt
    u = synth.make_uniforms(33, 4, 12)
    gpu.set_repeat_penalty(2.0)
    gpu.prefill(seqs)
    late = G.HipGpt(cfg, w, max_batch=4, max_seq_len=64)
    late.prefill(seqs)
    with pytest.raises(TSHipError, match="under way"):                  # the history cannot start in the middle of a sequence
        late.set_repeat_penalty(2.0)
    late.close()
    ids, _ = gpu.generate(8, mode=G.TOPP, top_p=0.95, temperature=1.0, uniforms=u[:8])
    cur = seqs
    want = []
    for s in range(12):
        p, _ = orc.step(cur, use_cache=True, sampling=True)
        nxt = oracle.toppsample(p, 0.95, 2.0, cur, u[s]).astype(np.int32)
        want.append(nxt)
        cur = np.concatenate([cur, nxt[:, None]], 1)
    want = np.stack(want)
    assert np.array_equal(ids, want[:8])
    # the penalty matters on this input
    orc.reset()
    p0, _ = orc.step(seqs, use_cache=True, sampling=True)
    differs = any(not np.array_equal(oracle.toppsample(p0, 0.95, 2.0, seqs, u[s]), oracle.toppsample(p0, 0.95, 0.0, None, u[s])) for s in range(12))
    assert differs
    # stepwise continuation: sample (no recording) then decode with the caller's tokens (recorded)
    for s in range(8, 12):
        t = gpu.sample(mode=G.TOPP, top_p=0.95, uniforms=u[s])
        assert np.array_equal(t, want[s])
        gpu.decode(t)
    # a new prompt after reset starts from an empty history
    gpu.reset()
    gpu.prefill(seqs)
    ids2, _ = gpu.generate(8, mode=G.TOPP, top_p=0.95, temperature=1.0, uniforms=u[:8])
    assert np.array_equal(ids2, want[:8])
    gpu.close()


@pytest.mark.parametrize("dtype,act", [("f32", synth.RELU), ("f32", synth.SILU), ("f16", synth.RELU)])
def test_moe_model(G, oracle, dtype, act):
    """MoE layers (layers >= 2): routing indices bit-exact on the fp32 model, logits within the dtype's bar."""
    cfg = synth.tiny_config(n_layers=4, n_experts=4, experts_per_token=2, norm_type=synth.LAYERNORM, act=act, dtype=dtype, batch=6)
    orc, gpu, out, cur = _teacher_forced(G, oracle, cfg, 31, 5)
    for lg, gl in out:
        if dtype == "f32":
            assert _rel(gl, lg) <= FP32_REL
        else:
            assert np.abs(gl - lg).max() <= FP16_ABS
    if dtype == "f32":
        ti, tv, pr = gpu.moe_routing(3)                      # the last MoE layer of the last step
        oi, ov, op = orc.moe_trace(1, cfg["batch"])
        assert np.array_equal(ti, oi)
        assert np.allclose(tv, ov, rtol=1e-6) and np.allclose(pr, op, rtol=1e-6)
    gpu.close()


@pytest.mark.parametrize("dtype,batch,prompt", [("f16", 4, 330), ("f16", 3, 70), ("f32", 2, 40)])
def test_moe_prefill_runs_the_experts_on_gathered_rows(G, oracle, monkeypatch, dtype, batch, prompt):
    """Prefill of a model with MoE layers: all prompt rows are routed at once, every expert runs the prefill GEMMs on the
    rows gathered for it (about 660 rows per expert in the first case: one launch for all experts; fewer than 512 in the
    others: one per expert), and the scaled outputs are added back in expert order.  Logits of the last position and the routing of the
    last position against the oracle, then decode steps on top of the cache the prefill wrote."""
    cfg = synth.tiny_config(n_layers=4, n_experts=4, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU, dtype=dtype,
                            batch=batch, prompt=prompt, vocab=300)      # (the third layer; the last one computes the last positions only)
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    orc, gpu, out, cur = _teacher_forced(G, oracle, cfg, 61, 3)
    kernels = gpu.profile_symbols()
    assert any("moe_lists_big_kernel" in s for s in kernels) and any("moe_gather_kernel" in s for s in kernels) == (batch * prompt < 512)
    for lg, gl in out:
        if dtype == "f32":
            assert _rel(gl, lg) <= FP32_REL
        else:
            assert np.abs(gl - lg).max() <= FP16_ABS
    if dtype == "f32":
        gpu.reset()
        gpu.prefill(cur)
        for layer in (2, 3):                                 # the last position of every sequence
            ti, tv, pr = gpu.moe_routing(layer)
            oi, ov, op = orc.moe_trace(layer - 2, batch)
            assert np.array_equal(ti, oi)
            assert np.allclose(pr, op, rtol=1e-6)
    gpu.close()


@pytest.mark.parametrize("batch,experts", [(70, 4), (50, 2), (100, 2)])
def test_moe_decode_batches_above_32_rows(G, oracle, batch, experts):
    """Decode with MoE layers and more than 32 rows (two and four 32-row tiles per block in the expert GEMMs): 70 rows over
    four experts; with two experts and two choices per token every expert gets all 50 or all 100 rows."""
    cfg = synth.tiny_config(n_layers=3, n_experts=experts, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU, dtype="f16",
                            batch=batch, prompt=5, vocab=200)
    orc, gpu, out, _ = _teacher_forced(G, oracle, cfg, 71, 3)
    for lg, gl in out:
        assert np.abs(gl - lg).max() <= FP16_ABS
    gpu.close()


def test_moe_tied_router_follows_topk_rule(G, oracle):
    cfg = synth.tiny_config(n_layers=3, n_experts=4, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU, batch=5)
    w = synth.make_weights(cfg, 41, random_bias=True)
    w["GPTDecoder.MoEFFN_2.m_Router"] = np.zeros_like(w["GPTDecoder.MoEFFN_2.m_Router"])
    w["GPTDecoder.MoEFFN_2.m_RouterBias"] = np.zeros_like(w["GPTDecoder.MoEFFN_2.m_RouterBias"])
    gpu = G.HipGpt(cfg, w, max_batch=5, max_seq_len=32)
    orc = oracle.OracleGpt(cfg, w)
    seqs = synth.make_prompts(cfg, 42)
    gpu.prefill(seqs)
    _, lg = orc.step(seqs, use_cache=True)
    ti, tv, pr = gpu.moe_routing(2)
    assert np.array_equal(ti, np.tile(np.array([0, 3], np.float32), (5, 1)))     # equal k-th entry is replaced by the later index
    assert np.array_equal(pr, np.full((5, 4), 0.25, np.float32))
    assert _rel(gpu.logits(), lg) <= FP32_REL
    gpu.close()


def test_full_width_layer_against_oracle(G, oracle):
    """The 1B configuration's layer shape (hidden 2048, 32/8 heads, FFN 5632 gated, RMSNorm) at 2 layers, batch 32:
    decode steps on the real decode kernels' tile shapes, checked against the oracle."""
    cfg = dict(synth.CONFIGS["cfg2_1b_gqa_f16"], n_layers=2, vocab=2048, batch=32, prompt=12)
    orc, gpu, out, _ = _teacher_forced(G, oracle, cfg, 61, 3)
    agree = []
    for lg, gl in out:
        assert np.abs(gl - lg).max() <= FP16_ABS
        agree.append((gl.argmax(1) == lg.argmax(1)).mean())
    assert np.mean(agree) >= 0.99
    gpu.close()


@pytest.mark.parametrize("kv_heads,batch,prompt", [(1, 3, 40), (2, 8, 70)])
def test_head_dim_128_against_oracle(G, oracle, kv_heads, batch, prompt):
    """The 7B configuration's head shape (head_dim 128, 4 or 2 query heads per KV head) on a narrow model: prefill
    (the second case has 560 prompt rows: MFMA prefill attention over several chunks) and decode
    steps across a 32-position chunk boundary, fp16, against the oracle."""
    cfg = synth.tiny_config(dtype="f16", hidden=512, n_heads=4, n_kv_heads=kv_heads, ffn_dim=1024, vocab=512, batch=batch, prompt=prompt)
    orc, gpu, out, _ = _teacher_forced(G, oracle, cfg, 71, 4)
    agree = []
    for lg, gl in out:
        assert np.abs(gl - lg).max() <= FP16_ABS
        agree.append(top1_agreement(gl, lg)[0])
    assert np.mean(agree) >= 0.99
    gpu.close()


@pytest.mark.parametrize("hidden,heads,kv_heads,batch,prompt,splits", [(256, 4, 2, 2, 300, 2), (512, 4, 1, 1, 200, 2), (256, 4, 4, 1, 530, 3),
                                                                      (256, 4, 2, 3, 90, 16), (1024, 16, 1, 1, 200, 2)])
def test_decode_attention_split_over_blocks(G, oracle, monkeypatch, hidden, heads, kv_heads, batch, prompt, splits):
    """Few (row, KV head) pairs and a long context: several blocks share a pair and the last one to arrive merges their
    sums.  The library only splits longer contexts; the environment variable forces it here
    (head_dim 64 and 128, two and three blocks, sixteen blocks most of which have no chunk at all, and sixteen query heads
    on one KV head, served as two groups of eight that each split in two).  fp16, against
    the oracle, with decode steps across a 32-position chunk boundary; then decode against the prefill path, which does
    not split."""
    monkeypatch.setenv("TSHIP_ATTN_SPLITS", str(splits))
    cfg = synth.tiny_config(dtype="f16", hidden=hidden, n_heads=heads, n_kv_heads=kv_heads, ffn_dim=2 * hidden, vocab=300, batch=batch, prompt=prompt)
    orc, gpu, out, cur = _teacher_forced(G, oracle, cfg, 81, 6)
    for lg, gl in out:
        assert np.abs(gl - lg).max() <= FP16_ABS
    # the same sequences through prefill only (one block per query group there)
    last = gpu.logits()
    gpu.reset()
    gpu.prefill(cur)
    assert np.abs(gpu.logits() - last).max() <= 2e-2
    gpu.close()


@pytest.mark.parametrize("hidden,heads,kv_heads,batch,at,cache", [(256, 4, 2, 1, 768, 1100), (256, 2, 1, 2, 640, 1100), (512, 8, 8, 5, 768, 1100),
                                                                  (512, 8, 8, 12, 960, 4100), (512, 4, 4, 25, 1152, 2100)])
def test_decode_attention_takes_more_blocks_as_the_context_grows(G, monkeypatch, hidden, heads, kv_heads, batch, at, cache):
    """Head sizes 64 and 128: the captured step goes on from the last position that one block of a pair takes by itself to the
    first that several share (the last two: two blocks, in caches long enough to launch them).  Against one block throughout, and
    against the prefill path."""
    cfg = synth.tiny_config(dtype="f16", hidden=hidden, n_heads=heads, n_kv_heads=kv_heads, ffn_dim=2 * hidden, vocab=300, batch=batch, prompt=at - 3)
    w = synth.make_weights(cfg, 83, random_bias=True)
    seqs = synth.make_prompts(cfg, 84)
    got = []
    for splits in (None, "1"):
        if splits:
            monkeypatch.setenv("TSHIP_ATTN_SPLITS", splits)
        gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=cache)
        gpu.prefill(seqs)
        ids, _ = gpu.generate(6)
        ids = ids.reshape(6, batch)
        gpu.set_seq_len(batch, at - 3)
        steps = []
        for i in range(6):
            gpu.decode(ids[i])
            steps.append(gpu.logits())
        got.append(steps)
        if not splits:
            first = ids
            gpu.reset()
            gpu.prefill(np.concatenate([seqs, ids.T], 1))
            assert np.abs(gpu.logits() - steps[-1]).max() <= 2e-2
        else:
            assert np.array_equal(ids, first)
        gpu.close()
    for a, b in zip(*got):      # (fp16 outputs of fp32 sums in another order)
        assert np.abs(a - b).max() <= 4e-3 * np.abs(b).max()
    assert np.array_equal(got[0][0], got[1][0]) and not np.array_equal(got[0][-1], got[1][-1])


@pytest.mark.parametrize("name,tiles", [("gqa_rms_gate", 20), ("gqa_rms_gate", 30), ("gqa_rms_gate_silu", 40), ("mha_ln_relu", 20),
                                        ("odd_sizes", 30), ("gqa_leaky_d32_g4", 40), ("gqa_rms_gate", 15), ("mha_ln_relu", 15),
                                        ("odd_sizes", 15), ("gqa_leaky_d32_g4", 15), ("gqa_rms_gate_silu", 15)])
def test_decode_ffn_up_projection_several_tiles_per_block(G, oracle, monkeypatch, name, tiles):
    """Decode, FFN up projection: a block takes several neighbouring 32-column tiles with one copy of the activations
    (the library does so when that shortens the busiest compute unit's work: more column tiles than compute units).  The
    environment variable forces two, three and four tiles (20, 30, 40) and a tile and a half (15: one tile plus the
    columns 0-7 / 16-23 or 8-15 / 24-31 of a neighbour) here: gated and plain activations, RMSNorm (deferred) and
    LayerNorm, and tile counts that are no multiple of the tiles per block (the last blocks then have fewer)."""
    monkeypatch.setenv("TSHIP_FFN_TILES", str(tiles))
    cfg = synth.tiny_config(dtype="f16", **TINY[name])
    orc, gpu, out, _ = _teacher_forced(G, oracle, cfg, 5, 5)
    for lg, gl in out:
        assert np.abs(gl - lg).max() <= FP16_ABS
    forced = [gl for _, gl in out]
    gpu.close()
    # one tile per block computes the same sums in the same order: bit-equal logits
    monkeypatch.setenv("TSHIP_FFN_TILES", "10")
    _, gpu, out, _ = _teacher_forced(G, oracle, cfg, 5, 5)
    for a, (_, b) in zip(forced, out):
        assert np.array_equal(a, b)
    gpu.close()


@pytest.mark.parametrize("dtype,hidden,heads,kv_heads,first,second", [("f32", 64, 4, 2, 5, 7), ("f16", 256, 4, 2, 64, 40), ("f16", 256, 4, 2, 45, 530),
                                                                    ("f16", 512, 4, 1, 32, 33)])
def test_prefill_appends_to_cached_sequences(G, oracle, dtype, hidden, heads, kv_heads, first, second):
    """A second prefill continues the cached sequences (the next turn of a dialogue whose cache was kept): the logits
    and the cache are those of one prefill of the concatenation, and decoding goes on from there.  Covers a first part
    that ends on a 32-position boundary (whole fragments written) and ones that do not, head_dim 64 and 128, and
    a second part of 530 x 2 rows."""
    cfg = synth.tiny_config(dtype=dtype, hidden=hidden, n_heads=heads, n_kv_heads=kv_heads, ffn_dim=2 * hidden, vocab=300, batch=2, prompt=first + second)
    w = synth.make_weights(cfg, 91, random_bias=True)
    orc = oracle.OracleGpt(cfg, w)
    seqs = synth.make_prompts(cfg, 92)
    gpu = G.HipGpt(cfg, w, max_batch=2, max_seq_len=first + second + 8)
    gpu.prefill(seqs)
    whole = gpu.logits()
    k_whole = gpu.get_kv(cfg["n_layers"] - 1, 0)
    gpu.reset()
    gpu.prefill(seqs[:, :first])
    gpu.prefill(seqs[:, first:])
    assert gpu.seq_len() == first + second
    tol = 1e-4 * float(np.abs(whole).max()) if dtype == "f32" else 2e-2
    assert np.abs(gpu.logits() - whole).max() <= tol
    assert np.abs(gpu.get_kv(cfg["n_layers"] - 1, 0) - k_whole).max() <= (1e-5 if dtype == "f32" else 2e-2)
    p, lg = orc.step(seqs, use_cache=True)
    assert np.abs(gpu.logits() - lg).max() <= (1e-4 * float(np.abs(lg).max()) if dtype == "f32" else FP16_ABS)
    nxt = oracle.argmax(p).astype(np.int32)
    p, lg = orc.step(np.concatenate([seqs, nxt[:, None]], 1), use_cache=True)
    gpu.decode(nxt)
    assert np.abs(gpu.logits() - lg).max() <= (1e-4 * float(np.abs(lg).max()) if dtype == "f32" else FP16_ABS)
    gpu.close()


def test_blocked_tokens(G, oracle):
    """Decoder.cs:745-753: probs += scatter(-1 at the blocked ids) before argmax / TopPSample."""
    cfg = synth.tiny_config(batch=4, vocab=120)
    w = synth.make_weights(cfg, 51, random_bias=True)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=4, max_seq_len=32)
    seqs = synth.make_prompts(cfg, 52)
    u = synth.make_uniforms(53, 4, 4)
    p, _ = orc.step(seqs, use_cache=True, sampling=True)
    blocked = np.unique(np.concatenate([oracle.argmax(p).astype(np.int32), np.argsort(-p[0])[:5].astype(np.int32)]))
    pm = p.copy()
    pm[:, blocked] = pm[:, blocked] + np.float32(-1.0)
    gpu.prefill(seqs)
    assert np.array_equal(gpu.sample(), oracle.argmax(p).astype(np.int32))
    gpu.set_blocked_tokens(blocked)
    got = gpu.sample()
    assert np.array_equal(got, oracle.argmax(pm).astype(np.int32)) and not np.isin(got, blocked).any()
    got = gpu.sample(mode=G.TOPP, top_p=0.9, uniforms=u[0])
    assert np.array_equal(got, oracle.toppsample(pm, 0.9, 0.0, None, u[0]).astype(np.int32))
    ids, _ = gpu.generate(4, mode=G.TOPP, top_p=0.9, uniforms=u)         # the graph loop sees the same list
    assert np.array_equal(ids[0], got) and not np.isin(ids, blocked).any()
    gpu.set_blocked_tokens([])
    gpu.reset()
    gpu.prefill(seqs)
    assert np.array_equal(gpu.sample(), oracle.argmax(p).astype(np.int32))
    gpu.close()


def test_generate_until_all_rows_emit_eos(G):
    """GPT.cs:299-302: the loop ends after the first step at which every sequence's newest token is the END tag
    (Decoder.cs:207-221); a row that ended earlier keeps generating until then."""
    cfg = synth.tiny_config(batch=3, vocab=50)
    w = synth.make_weights(cfg, 41)
    gpu = G.HipGpt(cfg, w, max_batch=3, max_seq_len=48)
    prompts = synth.make_prompts(cfg, 42)
    prompts[1] = prompts[0]
    prompts[2] = prompts[0]                                             # identical rows emit identical tokens
    gpu.prefill(prompts)
    full, _ = gpu.generate(20)
    assert np.array_equal(full[:, 0], full[:, 1])
    first = {}
    for s, tok in enumerate(full[:, 0]):
        first.setdefault(int(tok), s)
    eos, stop = max(first.items(), key=lambda kv: kv[1])                # the token whose first occurrence comes last
    assert stop >= 2
    gpu.reset()
    gpu.prefill(prompts)
    got, _ = gpu.generate_until(20, eos)
    assert got.shape[0] == stop + 1 and np.array_equal(got, full[:stop + 1])
    assert gpu.seq_len() == prompts.shape[1] + stop + 1
    rest, _ = gpu.generate(20 - stop - 1)                               # the state is that of the uninterrupted run
    assert np.array_equal(rest, full[stop + 1:])
    # rows that differ: one of them emitting the tag does not end the loop
    gpu.reset()
    prompts2 = synth.make_prompts(cfg, 43)
    gpu.prefill(prompts2)
    ref, _ = gpu.generate(12)
    col = ref[:, 0]
    others_differ = [s for s in range(12) if not (ref[s] == col[s]).all()]
    assert others_differ
    s0 = others_differ[0]
    all_same = [s for s in range(12) if (ref[s] == col[s0]).all()]
    gpu.reset()
    gpu.prefill(prompts2)
    got, _ = gpu.generate_until(12, int(col[s0]))
    assert got.shape[0] == (all_same[0] + 1 if all_same else 12) and np.array_equal(got, ref[:got.shape[0]])
    gpu.close()


def test_argument_errors(G):
    from seq2seqsharp_amd._lib import TSHipError
    cfg = synth.tiny_config()
    w = synth.make_weights(cfg, 0)
    gpu = G.HipGpt(cfg, w, max_batch=2, max_seq_len=12)
    with pytest.raises(TSHipError, match="out of range"):
        gpu.prefill(np.full((2, 4), cfg["vocab"], np.int32))
    with pytest.raises(TSHipError, match="batch"):
        gpu.prefill(np.zeros((3, 4), np.int32))
    gpu.prefill(synth.make_prompts(cfg, 1))
    with pytest.raises(TSHipError, match="max_seq_len"):
        gpu.generate(10)
    bad = dict(w)
    del bad["GPTDecoder.SelfAttn_1.W0"]
    with pytest.raises(TSHipError, match="never set"):
        G.HipGpt(cfg, bad, max_batch=2, max_seq_len=12)
    bad = dict(w, **{"GPTDecoder.SelfAttn_1.W0": np.zeros((3, 3), np.float32)})
    with pytest.raises(TSHipError, match="shape"):
        G.HipGpt(cfg, bad, max_batch=2, max_seq_len=12)
    gpu.close()


@pytest.mark.parametrize("experts,k,batch,prompt,router_bias", [
    (4, 1, 5, 520, None),                 # 2600 rows, one choice per token
    (16, 4, 2, 300, None),                # 600 rows, 2400 (token, choice) pairs over 16 experts: about 150 rows each
    (4, 2, 3, 200, (-60.0, 0.0, 0.0, 0.0)),       # expert 0 is never chosen: a problem with no rows
    (4, 2, 3, 200, (60.0, 0.0, 0.0, 0.0)),        # expert 0 is chosen by every token: all 600 rows in one problem
    (8, 2, 1, 777, None),                 # row counts that are no multiples of anything
])
def test_moe_prefill_one_launch_for_all_experts_equals_one_per_expert(G, oracle, monkeypatch, experts, k, batch, prompt, router_bias):
    """From 512 prompt rows on, the prefill of an fp16 model never reads the experts' row counts back: each projection of
    all experts is one launch of the 256 x 256 kernel over the experts' row tiles packed one behind the other (weights by
    pointer table, the problem of a tile found on the device from the counts), and the up projection reads its rows
    through the token lists.  Same logits, bit for bit, as the path with the counts on the host, gathered rows and one
    launch per expert (TSHIP_NO_MOE_BATCH=1): with an expert that holds far fewer rows than the largest one, one with no
    rows at all, one with every row, and row counts that fill no tile.  And the logits against the oracle.  (In the third layer of
    four: the keys and values of the last one follow from all its rows.)"""
    monkeypatch.setenv("TSHIP_RECORD_SYMBOLS", "1")
    cfg = synth.tiny_config(n_layers=4, n_experts=experts, experts_per_token=k, norm_type=synth.LAYERNORM, act=synth.RELU, dtype="f16",
                            batch=batch, prompt=prompt, vocab=300)
    w = synth.make_weights(cfg, 62, random_bias=True)
    if router_bias is not None:
        w = dict(w)
        w["GPTDecoder.MoEFFN_2.m_RouterBias"] = np.asarray(router_bias, np.float32).reshape(1, experts)
    seqs = synth.make_prompts(cfg, 162)
    gpu = G.HipGpt(cfg, w, max_batch=batch, max_seq_len=prompt + 10)
    gpu.prefill(seqs)
    one, cache = gpu.logits(), [gpu.get_kv(3, i) for i in range(2)]
    assert not any("moe_gather_kernel" in s for s in gpu.profile_symbols())
    if router_bias is not None:
        ti, _, _ = gpu.moe_routing(2)
        assert (ti == 0).any(axis=1).all() if router_bias[0] > 0 else not (ti == 0).any()
    monkeypatch.setenv("TSHIP_NO_MOE_BATCH", "1")
    gpu.reset()
    gpu.prefill(seqs)
    monkeypatch.delenv("TSHIP_NO_MOE_BATCH")
    assert any("moe_gather_kernel" in s for s in gpu.profile_symbols())
    assert np.array_equal(one, gpu.logits()) and all(np.array_equal(cache[i], gpu.get_kv(3, i)) for i in range(2))
    _, lg = oracle.OracleGpt(cfg, w).step(seqs, use_cache=True)
    assert np.abs(one - lg).max() <= FP16_ABS
    gpu.close()
