"""MoE prefills of several sizes on one model: the workspace of a prompt lies over the data of the one before."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_prompts_of_several_sizes(dtype):
    """Prompts behind larger and smaller ones, in all forms of the experts' projections (packed, one by one): the bits of a model that
    sees them first.  (Enough sizes that what a layout takes for granted lies in another's data.)"""
    from seq2seqsharp_amd import gpt as G
    cfg = synth.tiny_config(n_layers=4, n_experts=8, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU, dtype=dtype, vocab=300)
    w = dict(synth.make_weights(cfg, 62, random_bias=True))
    for name in w:
        if "MoEFFN" in name and "m_Whd" in name:
            w[name] = w[name] * np.float32(8)      # (outputs of the size of the residual stream)

    def run(gpu, seqs):
        gpu.reset()
        gpu.prefill(seqs)
        return [gpu.logits()] + [gpu.get_kv(l, i) for l in range(4) for i in range(2)]

    used = G.HipGpt(cfg, w, max_batch=3, max_seq_len=310)
    for n in (20, 300, 270, 240, 210, 190, 175, 150, 130, 110, 90, 70, 60, 41, 33, 20, 300):
        seqs = synth.make_prompts(cfg, 7 + n, batch=3, length=n)
        fresh = G.HipGpt(cfg, w, max_batch=3, max_seq_len=310)
        for a, b in zip(run(used, seqs), run(fresh, seqs)):
            assert np.array_equal(a, b), n
        fresh.close()
    used.close()
