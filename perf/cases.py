"""Timed workloads of the GPT decoder path: what a program that serves these models has the library do.

Every case is one pass through `HipGpt`, the host side of the library: prompts, turns of a conversation, token loops
(greedy and top-p) and beam search, on the model shapes of `seq2seqsharp_amd.synth`.  A pass starts from sequences that
the state's cache already holds (`context` tokens each) or from an empty cache, feeds the pass's tokens and returns the
new token ids and the logits of the last step on the host, as the library's calls deliver them.

The weights are random, of the sizes of real models, with two properties of trained ones that keep greedy choices and
expert choices well apart from their runners-up: the vocabulary projection is tied to the embedding (the model is sure of
its next token, here the current one plus a constant), and the experts' router is decided.  Without them a choice between
two equal logits would turn on the last bit of a sum.
"""
import math

import numpy as np
import torch

from seq2seqsharp_amd import synth
from seq2seqsharp_amd.gpt import GREEDY, TOPP, HipGpt

# The model shapes of the benchmark configurations.  The 7B one keeps 8 of its 32 equal layers, so that a state is made in
# a second; a layer's work and the context it meets stay those of the whole model.
MODELS = {
    "tiny_mha_f32": synth.CONFIGS["cfg0_tiny_mha_f32"],
    "gpt2small_f32": synth.CONFIGS["cfg1_gpt2small_f32"],
    "gpt2small_f16": synth.CONFIGS["cfg1_gpt2small_f16"],
    "1b_gqa_f16": synth.CONFIGS["cfg2_1b_gqa_f16"],
    "moe_f16": synth.CONFIGS["cfg3_moe_f16"],
    "7b_gqa_f16": dict(synth.CONFIGS["cfg4_7b_longctx_f16"], n_layers=8),
}
NEXT_TOKEN = 4099          # the tied projection favours the current token plus this
EMBEDDING_STD = 0.04
ROUTER_GAIN = 8.0
EOS = 0


def _case(name, model, batch, context, prompt, steps, padded=False, top_p=0.0, penalty=0.0, beam=0):
    case = dict(model=model, batch=batch, context=context, prompt=prompt, steps=steps, padded=padded, top_p=top_p, penalty=penalty, beam=beam)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # one user, a small fp32 model: a call is a handful of microseconds of work per layer, launches and latency are all of it
        _case("chat_tiny_f32", "tiny_mha_f32", 1, 64, 0, 32),
        # translation-style beam search on an fp32 model: two prompts, four hypotheses each
        _case("beam_gpt2small_f32", "gpt2small_f32", 2, 0, 300, 8, beam=4),
        # a small fp16 LayerNorm model behind a service: eight sequences, token loop
        _case("decode_gpt2small_f16", "gpt2small_f16", 8, 512, 0, 32),
        # one user's next turn with a 1B model: 37 new tokens behind a kept conversation, then the answer
        _case("chat_turn_1b", "1b_gqa_f16", 1, 1000, 37, 16),
        # the benchmark's token loop: 1B model, 32 sequences at a context of 1024
        _case("decode_1b_b32", "1b_gqa_f16", 32, 1024, 0, 16),
        # the same model behind a busier service, more sequences than one tile of 32 rows
        _case("decode_1b_b96", "1b_gqa_f16", 96, 300, 0, 8),
        # whole requests sampled with top-p and the reference's default repeat penalty: prompt in, 24 tokens out
        _case("sampled_request_1b", "1b_gqa_f16", 16, 0, 100, 24, top_p=0.9, penalty=2.0),
        # mixture of experts, whole requests: prompts of 64 sequences, then the token loop
        _case("request_moe", "moe_f16", 64, 0, 256, 16),
        # long context: 16 sequences of 8k tokens, token loop (attention reads the cache)
        _case("decode_7b_8k", "7b_gqa_f16", 16, 8192, 0, 4),
        # a full batch of prompts at once (the benchmark's prefill)
        _case("prefill_1b_32x1024", "1b_gqa_f16", 32, 0, 1024, 0),
        # a small ragged batch, padded to its longest prompt: odd row counts, the reference's masking of padded batches
        _case("prefill_1b_ragged", "1b_gqa_f16", 5, 0, 333, 0, padded=True),
        # one long document: attention is a large share of the work
        _case("prefill_7b_8k", "7b_gqa_f16", 1, 0, 8000, 0),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed kinds, sizes spread over the range each kind stands for."""
    kind = rng.choice(["decode", "decode", "decode", "turn", "request", "sampled", "prefill", "prefill", "padded", "beam"])
    if kind == "beam":
        model = rng.choice(["tiny_mha_f32", "gpt2small_f32"])
        return _case("", model, rng.randint(1, 3), 0, _log_int(rng, 150, 500), rng.randint(3, 8), beam=rng.randint(2, 4))
    if kind in ("prefill", "padded"):
        model = rng.choice(["gpt2small_f32", "gpt2small_f16", "1b_gqa_f16", "1b_gqa_f16", "moe_f16", "7b_gqa_f16"])
        rows = _log_int(rng, 40, {"gpt2small_f32": 4096, "7b_gqa_f16": 8192}.get(model, 32768))
        batch = max(1, min(_log_int(rng, 1, 32), rows // 20))
        if kind == "padded":
            batch = max(batch, 2)
        return _case("", model, batch, 0, min(rows // batch, 8192), 0, padded=kind == "padded")
    if kind == "sampled":
        return _case("", rng.choice(["gpt2small_f16", "1b_gqa_f16"]), _log_int(rng, 1, 32), 0, _log_int(rng, 20, 400), rng.randint(8, 24),
                     top_p=rng.choice([0.8, 0.9, 0.95]), penalty=rng.choice([0.0, 2.0]))
    if kind == "request":
        model = rng.choice(["moe_f16", "moe_f16", "1b_gqa_f16"])
        return _case("", model, _log_int(rng, 1, 64), 0, _log_int(rng, 20, 300), rng.randint(4, 16))
    if kind == "turn":
        return _case("", rng.choice(["gpt2small_f16", "1b_gqa_f16", "moe_f16"]), rng.choice([1, 1, 2, 3, 6]), _log_int(rng, 100, 2000), _log_int(rng, 8, 200), rng.randint(8, 24))
    model = rng.choice(["tiny_mha_f32", "gpt2small_f32", "gpt2small_f16", "1b_gqa_f16", "1b_gqa_f16", "moe_f16", "7b_gqa_f16"])
    batch = _log_int(rng, 1, {"7b_gqa_f16": 16, "tiny_mha_f32": 8, "gpt2small_f32": 16}.get(model, 128))
    context = _log_int(rng, 30, {"7b_gqa_f16": 8192, "tiny_mha_f32": 500}.get(model, 2000))
    if batch * context > 131072:
        context = 131072 // batch
    return _case("", model, batch, context, 0, rng.randint(4, 16))


def _weights(cfg, seed):
    """(name, host float32 array) in the order of the parameter list.  The normal weights are stretches of one noise tensor made
    on the GPU, at places of their own, so that a model of a billion parameters is made in a fraction of a second."""
    shapes = synth.weight_shapes(cfg)
    largest = max(math.prod(s) for _, s, _ in shapes)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    noise = torch.randn(largest + (1 << 22), device="cuda", generator=gen) * 0.02
    if cfg["dtype"] == "f16":
        noise = noise.half().float()
    host = torch.empty(noise.numel(), pin_memory=True)
    host.copy_(noise)
    vocab, hidden = cfg["vocab"], cfg["hidden"]
    table = noise[:vocab * hidden].view(vocab, hidden) * (EMBEDDING_STD / 0.02)
    spare = torch.empty(vocab * hidden, pin_memory=True)
    at = 0
    for name, shape, kind in shapes:
        n = math.prod(shape)
        if name == "TgtEmbeddings":
            spare.copy_(table.reshape(-1))
            yield name, spare.numpy().reshape(shape)
        elif name == "FeedForward_Decoder_0.m_Whd":      # column v: the embedding of token v - NEXT_TOKEN
            spare.copy_(table.roll(NEXT_TOKEN, 0).t().reshape(-1))
            yield name, spare.numpy().reshape(shape)
        elif kind == "normal":
            at = (at + 7919 * 64 + 64 * int(rng.integers(0, 4096))) % (1 << 22)
            w = host[at:at + n].numpy().reshape(shape)
            yield name, w * np.float32(ROUTER_GAIN) if name.endswith("m_Router") else w
        elif kind == "ones":
            yield name, (1.0 + 0.1 * rng.standard_normal(shape)).astype(np.float32)
        else:
            yield name, (0.02 * rng.standard_normal(shape)).astype(np.float32)


def _ids(rng, cfg, batch, length):
    return rng.integers(4, cfg["vocab"], size=(batch, length), dtype=np.int32)


def prepare(case, seed):
    cfg = MODELS[case["model"]]
    rng = np.random.default_rng(seed + 1)
    rows = case["batch"] * max(1, case["beam"])
    total = case["context"] + max(1, case["prompt"]) + case["steps"] + 1
    model = HipGpt(cfg, _weights(cfg, seed), max_batch=rows, max_seq_len=total)
    if case["penalty"]:
        model.set_repeat_penalty(case["penalty"])
    if case["context"]:
        model.prefill(_ids(rng, cfg, case["batch"], case["context"]))      # the conversation so far
    state = dict(case=case, model=model, ids=_ids(rng, cfg, case["batch"], max(1, case["prompt"])), lens=None, uniforms=None)
    if case["padded"]:
        lens = rng.integers(max(1, case["prompt"] // 3), case["prompt"] + 1, size=case["batch"])
        lens[rng.integers(0, case["batch"])] = case["prompt"]
        state["ids"], state["lens"] = HipGpt.pad_sentences([row[:n] for row, n in zip(state["ids"], lens)], pad_id=EOS)
    if case["top_p"]:
        state["uniforms"] = synth.make_uniforms(seed + 2, case["batch"], case["steps"])
    return state


def run(state):
    case, model = state["case"], state["model"]
    if case["beam"]:
        hypotheses, scores = model.beam_search(state["ids"], case["beam"], case["prompt"] + case["steps"], eos_id=EOS)
        return np.array(hypotheses, np.int32), np.array(scores, np.float32), model.logits()
    if case["context"]:
        model.set_seq_len(case["batch"], case["context"])      # back to the end of the kept conversation
    else:
        model.reset()
    if case["prompt"]:
        model.prefill(state["ids"], state["lens"])
    else:
        model.decode(state["ids"])
    if case["top_p"]:
        ids, _ = model.generate(case["steps"], TOPP, case["top_p"], 1.0, state["uniforms"])
    elif case["steps"]:
        ids, _ = model.generate(case["steps"], GREEDY)
    else:
        ids = model.sample(GREEDY)
    return ids, model.logits()


def work(case):
    """Bytes and operations of a pass: a prompt reads the weights and the cache in front of it once and writes its keys and
    values; every token of the loop depends on the one before, so it reads the weights (of a mixture of experts: those of the
    experts that the batch is expected to hit), the whole cache and writes the logits once more."""
    c = MODELS[case["model"]]
    size = 2 if c["dtype"] == "f16" else 4
    h, layers, vocab, heads = c["hidden"], c["n_layers"], c["vocab"], c["n_heads"]
    d, kv_heads = h // heads, c["n_kv_heads"]
    n_experts, top = c["n_experts"], c["experts_per_token"]
    n_moe = max(layers - 2, 0) if n_experts > 1 else 0
    attn = h * (heads + 2 * kv_heads) * d + h * h
    ffn = h * c["ffn_dim"] * (3 if c["act"] in (synth.SWIGLU, synth.SWIGLU_SILU) else 2)
    expert = 8 * h * h
    kv = layers * 2 * kv_heads * d * size                  # bytes of one position
    params_row = layers * attn + (layers - n_moe) * ffn + n_moe * (top * expert + h * n_experts)      # without the vocabulary projection

    def params_read(rows):
        hit = n_experts * (1.0 - (1.0 - top / n_experts) ** rows) if n_moe else 0
        return layers * attn + (layers - n_moe) * ffn + n_moe * (hit * expert + h * n_experts)

    n_bytes = n_flops = 0.0

    def feed(rows, new, before):
        nonlocal n_bytes, n_flops
        tokens = rows * new
        seen = new * before + new * (new + 1) / 2          # (query, key) pairs of a row
        n_bytes += size * (params_read(tokens) + h * vocab + tokens * h) + rows * (before + new) * kv + rows * vocab * 4
        n_flops += 2.0 * tokens * params_row + 2.0 * rows * h * vocab + 4.0 * rows * layers * heads * d * seen

    batch = case["batch"]
    feed(batch, max(1, case["prompt"]), case["context"])
    at = case["context"] + max(1, case["prompt"])
    loop = max(0, case["steps"] - 1) if case["beam"] else case["steps"]      # (beam search ends on a choice, without a step behind it)
    for i in range(loop):
        feed(batch * max(1, case["beam"]), 1, at + i)
    return {"bytes": n_bytes, "flops": n_flops}


def tolerance(case):
    """Four times what was measured between two orders of the same sums: fp16 models with other row tiles, K splits and prefill
    kernels 0.9e-3 to 1.3e-3 (largest single difference 8e-3), fp32 models against a CPU evaluation 1.0e-6 (4.5e-6).  A router
    logit on the edge of its rounding step can send a row to another second expert, which moves that row's logits by some
    hundredths of the logits' size.  A token may differ where two logits tie."""
    if MODELS[case["model"]]["dtype"] == "f32":
        return {"rel": 4e-6, "max": 2e-5, "differ": 0.005}
    if MODELS[case["model"]]["n_experts"] > 1:
        return {"rel": 8e-3, "max": 0.2, "differ": 0.005}
    return {"rel": 5e-3, "max": 3e-2, "differ": 0.005}
