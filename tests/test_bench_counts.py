"""The operations bench.py credits a prefill with are those that are done for its result."""
import pytest

from bench import algorithmic_prefill_flops
from seq2seqsharp_amd import synth


@pytest.mark.parametrize("name", ["cfg1_gpt2small_f16", "cfg2_1b_gqa_f16", "cfg3_moe_f16", "cfg4_7b_longctx_f16"])
@pytest.mark.parametrize("batch,prompt", [(32, 1024), (3, 200)])
def test_prefill_operations(name, batch, prompt):
    """Against a count that walks back from the logits: a layer's rows behind its queries, keys and values are those that the layer above it reads."""
    c = synth.CONFIGS[name]
    h, d = c["hidden"], c["hidden"] // c["n_heads"]
    kv_columns = 2 * c["n_kv_heads"] * d
    total, needed = 2.0 * batch * h * c["vocab"], 1          # (positions of a sequence whose output is read)
    for layer in reversed(range(c["n_layers"])):
        if c["n_experts"] > 1 and layer > 1:
            ffn = c["experts_per_token"] * 8 * h * h + h * c["n_experts"]
        else:
            ffn = (3 if c["act"] in (synth.SWIGLU, synth.SWIGLU_SILU) else 2) * h * c["ffn_dim"]
        pairs = prompt if needed == 1 else prompt * (prompt + 1) / 2
        total += 2.0 * batch * (needed * (h * h + ffn) + prompt * h * (h + kv_columns)) + 4.0 * batch * h * pairs
        needed = prompt                                      # every position's keys and values are read
    assert algorithmic_prefill_flops(c, batch, prompt) == pytest.approx(total, rel=2e-3)
