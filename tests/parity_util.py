"""Shared assertions of the parity tests."""
import numpy as np


def top1_agreement(gl, lg):
    """Per-row top-1 agreement of device logits `gl` with oracle logits `lg`.  A row whose winner differs is a tie
    (counted as agreeing) when the oracle's own gap between its winner and the device's winner is within twice that
    row's largest logit error: the device cannot separate two candidates closer than its own error, and the contract's
    99 % bar is about mistakes, not about coin flips between equals.  Returns (fraction with ties counted, strict)."""
    a, b = gl.argmax(1), lg.argmax(1)
    rows = np.arange(lg.shape[0])
    gap = lg[rows, b] - lg[rows, a]
    err = np.abs(gl - lg).max(1)
    ok = (a == b) | (gap <= 2.0 * err)
    return float(ok.mean()), float((a == b).mean())


# fp16 logits of models with `sensitive` weights: largest difference over the largest logit.  The device's error is a few
# roundings to 16 bits per layer (2^-11 of a value each, 1e-3 to 3e-3 of the largest logit in sum); a projection that returned
# zero moves the logits by 9e-2 and more (test_parity_bars.py).
FP16_SENSITIVE_REL = 1e-2


def sensitive(w, hidden):
    """The weights of a tiny model scaled so that every projection counts: queries and keys that make attention far from
    uniform, and values, output and feed-forward projections of about unit gain."""
    qk, rest = np.float32(62.0 / np.sqrt(hidden)), np.float32(26.0 / np.sqrt(hidden))
    out = dict(w)
    for name, x in w.items():
        if name.endswith((".Q", ".K")):
            x = x * qk
        elif name.endswith(".QKV"):
            x = np.concatenate([x[:, :2 * hidden] * qk, x[:, 2 * hidden:] * rest], 1)
        elif name.endswith((".V", ".W0")) or ("feedForwardLayer" in name and name.endswith("m_Whd")):
            x = x * rest
        out[name] = x.astype(np.float16).astype(np.float32)
    return out
