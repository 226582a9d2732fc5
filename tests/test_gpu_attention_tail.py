"""A prompt's attention where one key takes almost all of the weight: the many small weights beside it.

Trained models park most of a query's weight on the first token.  What the thousands of others add is then a
sum of weights around 1e-6, which has to keep its value.  Models of two layers with weights set by hand: the
first token's key scores `score` above all others (which score 0) and its value is 0, every other value is 1,
so the first layer's attention is the tail's mass n w / (1 + n w), w = exp(-score).  The output projection
adds it to a feature of the hidden row of its own, which the second layer's key row returns.

The bar of 1e-3 is one binary16 step of that cache row (2^-10); everything before it is binary32.
"""
import sys

import numpy as np
import pytest

from zhip import gguf, hip, synth
from zhip.gguf import F32

pytestmark = pytest.mark.gpu

FIRST, OTHER = 3, 4
GAIN = 4096.0


def build(hd, heads, score, context):
    spec = synth.small_spec(n_head=heads, n_kv=1, head_dim=hd, default_type=F32, attn_v_type=F32, output_type=F32,
                            embd_type=F32, context=context, rope_theta=1e30)
    h, d = spec.hidden, hd - 2  # RoPE at this base leaves the last dims of a head as they are
    mats = {t.name: np.zeros((t.rows, t.row_len), np.float32) for t in spec.tensors()}
    for name, m in mats.items():
        if name.endswith("_norm.weight"):
            m[:] = 1.0
    mats["token_embd.weight"][FIRST, 0] = mats["token_embd.weight"][OTHER, 1] = 16.0  # RMS 1
    for i in range(heads):
        mats["blk.0.attn_q.weight"][i * hd + d, 1] = 0.5
    mats["blk.0.attn_k.weight"][d, 0] = score * np.sqrt(hd) / 8.0 / 16.0
    mats["blk.0.attn_v.weight"][0, 1] = 1.0 / 16.0
    mats["blk.0.attn_output.weight"][2, 0] = GAIN  # the first head's dim 0 into feature 2
    mats["blk.1.attn_k.weight"][d, 2] = 1.0
    img = gguf.layout(spec.metadata(), spec.tensors())
    for name, m in mats.items():
        img.tensor_view(name)[:] = np.ascontiguousarray(m).reshape(-1).view(np.uint8)
    return spec, img, d


def want_tail(spec, hd, score, p):
    """The second layer's key entry of position p in 64 bits."""
    one = 16.0 / np.sqrt(256.0 / spec.hidden + spec.eps)  # the normed feature
    q = one * 0.5
    k = float(np.float16(one * score * np.sqrt(hd) / 8.0 / 16.0))
    w = np.exp(-q * k / np.sqrt(hd))
    hid = GAIN * p * w / (1.0 + p * w)
    return hid / np.sqrt((256.0 + hid * hid) / spec.hidden + spec.eps)


@pytest.mark.parametrize("score", [11.5, 13.75, 16.0])
@pytest.mark.parametrize("hd,heads", [(64, 8), (96, 2), (128, 4)])
# rows of the first turn and of the second (0: none): one pass whole, and short turns whose positions are
# split over 8 workgroups and over 16
@pytest.mark.parametrize("first,second", [(250, 0), (2100, 18), (4300, 40)])
def test_small_weights_beside_a_dominant_key(hip_ctx, hd, heads, score, first, second):
    print(f"attention tail hd {hd} score {score} rows {first}+{second}", flush=True)
    sys.stdout.flush()
    spec, img, d = build(hd, heads, score, 4400)
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate([FIRST] + [OTHER] * (first - 1), 0)
    if second:
        s.generate([OTHER] * second, 0)
    n = first + second
    # rows of the last pass (a prompt's last token runs through the decode step)
    for p in (n - 2, n - 3, max(first, n - 17)) if second else (n - 2, 130, 100, 17):
        got, want = float(s.kv(1, p)[0][d]), want_tail(spec, hd, score, p)
        assert abs(got - want) < 1e-3 * want, (p, got, want)
    s.close()
