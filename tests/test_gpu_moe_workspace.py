"""MoE prefills of several sizes on one model: the workspace of a prompt lies over the data of the one before."""
import numpy as np
import pytest

from seq2seqsharp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("first,second", [((3, 300), (2, 32)), ((3, 300), (3, 180)), ((2, 100), (2, 20)), ((2, 20), (3, 300))])
def test_prompts_of_several_sizes(dtype, first, second):
    """A prompt behind a larger (or smaller) one, in all forms of the experts' projections (packed, one by one): the bits of a model that sees it first."""
    from seq2seqsharp_amd import gpt as G
    cfg = synth.tiny_config(n_layers=4, n_experts=8, experts_per_token=2, norm_type=synth.LAYERNORM, act=synth.RELU, dtype=dtype, vocab=300)
    w = dict(synth.make_weights(cfg, 62, random_bias=True))
    for name in w:
        if "MoEFFN" in name and "m_Whd" in name:
            w[name] = w[name] * np.float32(8)      # (outputs of the size of the residual stream)
    prompts = [synth.make_prompts(cfg, 7 + i, batch=b, length=n) for i, (b, n) in enumerate((first, second))]

    def run(order):
        gpu = G.HipGpt(cfg, w, max_batch=3, max_seq_len=310)
        for seqs in order:
            gpu.reset()
            gpu.prefill(seqs)
        out = [gpu.logits()] + [gpu.get_kv(l, i) for l in range(4) for i in range(2)]
        gpu.close()
        return out

    for a, b in zip(run(prompts), run(prompts[1:])):
        assert np.array_equal(a, b)
