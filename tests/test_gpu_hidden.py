"""TSHip_GptGetHidden behind a prefill, a turn's second prefill and a decode step, against the oracle, on every form of the norms."""
import numpy as np
import pytest

from parity_util import FP16_SENSITIVE_REL, sensitive
from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,norm,experts,max_batch,batch,prompt", [
    ("f16", synth.LAYERNORM, 1, 3, 3, 7), ("f16", synth.LAYERNORM, 1, 5, 5, 128), ("f16", synth.LAYERNORM, 1, 40, 2, 9),      # LayerNorm: folded up to 32 rows, stored
    ("f16", synth.RMSNORM, 1, 3, 3, 7), ("f16", synth.RMSNORM, 1, 5, 5, 128), ("f16", synth.RMSNORM, 1, 40, 33, 9),
    ("f16", synth.LAYERNORM, 4, 3, 3, 7), ("f32", synth.RMSNORM, 1, 3, 3, 7), ("f32", synth.LAYERNORM, 4, 3, 3, 7)])
def test_hidden_state(oracle, dtype, norm, experts, max_batch, batch, prompt):
    from seq2seqsharp_amd import gpt as G
    cfg = synth._cfg(n_layers=3 if experts > 1 else 2, hidden=192, n_heads=3, n_kv_heads=3, ffn_dim=256, vocab=157, attn_type=synth.GQA, norm_type=norm, act=synth.RELU,
                     n_experts=experts, experts_per_token=min(2, experts), batch=batch, prompt=prompt, steps=2, dtype=dtype)
    w = synth.make_weights(cfg, 95, random_bias=True)
    if experts == 1:
        w = sensitive(w, 192)
    seqs = synth.make_prompts(cfg, 96)
    orc = oracle.OracleGpt(cfg, w)
    gpu = G.HipGpt(cfg, w, max_batch=max_batch, max_seq_len=prompt + 8)

    def check(want):
        assert np.abs(gpu.hidden() - want).max() <= (1e-4 if dtype == "f32" else FP16_SENSITIVE_REL) * np.abs(want).max()

    whole = orc.step(seqs, use_cache=True, want_hidden=True)[2]
    for cut in (prompt, 3):
        gpu.reset()
        gpu.prefill(seqs[:, :cut])
        if cut < prompt:
            gpu.prefill(seqs[:, cut:])
        check(whole)
    more = (np.arange(batch) + 5).astype(np.int32)
    gpu.decode(more)
    check(orc.step(np.concatenate([seqs, more[:, None]], 1), use_cache=True, want_hidden=True)[2])
    gpu.close()
