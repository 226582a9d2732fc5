"""The prompt products' running unit over a long reduction.

The accumulators are in units of the current block's scale and are multiplied by a rounded quotient at each
change of it: 448 times over 14336 Q8_0 values.  Scales that alternate repeat the same two quotients, whose
roundings must not add up.  Value rows whose second half takes back what the first half adds, but for eight
codes of the last block, show such a drift about a thousand times enlarged.

The bar, of the root mean square over 2048 rows: each of the 448 blocks rounds a sum that goes up to S and back
(mean square S^2 / 3) five times (the factor, and two products of two pieces), each by at most 2^-24 / sqrt(3)
of it, so 9.4e-7 S, where the result is about 1.1e-3 S; three times that, and the cache's binary16 (2^-11).
"""
import numpy as np
import pytest

from zhip import gguf, hip, synth
from zhip.gguf import Q8_0

pytestmark = pytest.mark.gpu


def test_alternating_scales_do_not_drift(hip_ctx):
    n, kv, rows = 14336, 2048, 2100  # rows x matrix rows past the split workspace: one reduction over all of it
    print("prompt units, alternating scales", flush=True)
    spec = synth.small_spec(n_layers=1, hidden=n, ffn=256, n_head=16, n_kv=16, head_dim=128, vocab=64,
                            default_type=Q8_0, attn_v_type=Q8_0, output_type=Q8_0, embd_type=Q8_0, context=2176)
    img = synth.build(spec, seed=5)
    rng = np.random.default_rng(6)
    nb = n // 32
    codes = rng.integers(64, 128, (kv, nb // 2, 32)).astype(np.int8)
    codes = np.concatenate([codes, -codes], 1)
    codes[:, -1, :8] = 0
    # a scale for the even blocks of a row and one for the odd
    d = np.tile((0.02 / 73 * (0.75 + 0.5 * rng.random((kv, 2)))).astype(np.float16), nb // 2)
    blocks = np.concatenate([d.view(np.uint8).reshape(kv, nb, 2), codes.view(np.uint8)], 2)
    img.tensor_view("blk.0.attn_v.weight")[:] = blocks.reshape(-1)
    emb = img.tensor_view("token_embd.weight").reshape(spec.vocab, nb, 34)
    emb[3, :, :2] = np.float16(1.0).reshape(1).view(np.uint8)
    emb[3, :, 2:] = 1
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate([3] * (rows + 1), 0)
    x = 1.0 / np.sqrt(1.0 + spec.eps)
    want = (codes.astype(np.float64).sum(2) * d.astype(np.float64)).sum(1) * x
    for p in (0, 1000, rows - 1):
        err = (s.kv(0, p)[1].astype(np.float64) - want) / want
        rms = np.sqrt((err ** 2).mean())
        assert rms < 3 * 9.4e-7 / 1.1e-3 + 2.0 ** -11
    s.close()
