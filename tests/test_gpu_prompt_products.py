"""Prompt passes' products (zh_pgemm.hip) in every format, at the edges of their tiles.

A prompt's rows run through the products as tiles of 64, 128 or 256 tokens with the reduction split where
few tiles would leave the chip idle.  Each model has one weight format, row counts off the 64- and 128-row
tiles, and reductions of an even and an odd number of 256-value blocks; the prompts end one row before, on
and after a tile's edge.  Logits within 1e-4 relative L2 and K/V rows within 1e-3 (one binary16 step) of
the oracle's token-by-token prompt, as in test_gpu_prefill.py.
"""
import sys

import numpy as np
import pytest

from oracle import zo
from zhip import hip, synth
from zhip.gguf import IQ4_XS, Q3_K, Q4_K, Q6_K, Q8_0, TYPE_NAMES

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("ttype", [Q4_K, Q6_K, Q8_0, IQ4_XS, Q3_K], ids=lambda t: TYPE_NAMES[t])
# n rows in the pass: prompt - 1
@pytest.mark.parametrize("rows", [17, 64, 65, 129, 257])
def test_prompt_rows_match_the_token_by_token_prompt(hip_ctx, ttype, rows):
    print(f"prompt products {TYPE_NAMES[ttype]} rows {rows}", flush=True)
    sys.stdout.flush()
    spec = synth.small_spec(hidden=512, ffn=768, n_head=4, n_kv=1, head_dim=64 if ttype == Q4_K else 128,
                            default_type=ttype, attn_v_type=ttype, output_type=Q8_0, embd_type=Q8_0, context=300)
    spec.n_head = 512 // spec.head_dim
    img = synth.build(spec, seed=17)
    prompt = synth.prompt_tokens(rows, rows + 1, spec.vocab)
    o = zo.Session(zo.Model(img.buf), context=spec.context, kv_f16=True)
    for t in prompt[:-1]:
        o.step_no_output(int(t))
    want = o.step(int(prompt[-1]))
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate(prompt, 0)
    assert rel_l2(s.logits(), want) < 1e-4
    for pos in (0, rows // 2, rows - 1):
        for a, b in zip(s.kv(1, pos), o.kv(1, pos)):
            assert rel_l2(a, b) < 1e-3
    s.close()


# heads, kv heads, head size: query heads per kv head 8, 1, 3 (126 of a workgroup's 128 rows) and 4
@pytest.mark.parametrize("heads,kv,hd", [(8, 1, 64), (4, 4, 128), (6, 2, 128), (8, 2, 96)])
@pytest.mark.parametrize("second", [18, 90])
def test_second_turn_attends_to_the_first(hip_ctx, heads, kv, hd, second):
    """A short turn after a long one: its positions are split over workgroups whose partial results merge,
    and its tiles start inside a page.  The bar is as above."""
    print(f"second turn {heads}/{kv} heads of {hd}, {second} rows", flush=True)
    spec = synth.small_spec(hidden=768, ffn=512, n_head=heads, n_kv=kv, head_dim=hd, default_type=Q8_0,
                            attn_v_type=Q8_0, output_type=Q8_0, embd_type=Q8_0, context=700)
    img = synth.build(spec, seed=23)
    first, then = synth.prompt_tokens(1, 590, spec.vocab), synth.prompt_tokens(2, second, spec.vocab)
    o = zo.Session(zo.Model(img.buf), context=spec.context, kv_f16=True)
    for t in [*first, *then[:-1]]:
        o.step_no_output(int(t))
    want = o.step(int(then[-1]))
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate(first, 0)
    s.generate(then, 0)
    assert rel_l2(s.logits(), want) < 1e-4
    for pos in (590, 590 + second // 2, 590 + second - 2):
        for a, b in zip(s.kv(1, pos), o.kv(1, pos)):
            assert rel_l2(a, b) < 1e-3
    s.close()


@pytest.mark.parametrize("ttype", [Q4_K, Q6_K, Q8_0, IQ4_XS, Q3_K], ids=lambda t: TYPE_NAMES[t])
def test_largest_tiles_match_the_step_path(hip_ctx, ttype):
    """4096-row matrices and 3841 prompt rows: tiles of 256 x 256, the last of them one row (gate and up, of 512
    rows, take smaller ones; test_tiles_and_splits_match_the_step_path has theirs).  Against the same
    prompt token by token through the decode step, which has the oracle's bars of 1e-4 and 1e-3: twice those."""
    print(f"largest tiles {TYPE_NAMES[ttype]}", flush=True)
    spec = synth.small_spec(hidden=4096, ffn=512, n_head=32, n_kv=32, head_dim=128, default_type=ttype,
                            attn_v_type=ttype, output_type=Q8_0, embd_type=Q8_0, context=3904)
    img = synth.build(spec, seed=29)
    prompt = synth.prompt_tokens(3, 3842, spec.vocab)
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate(prompt, 0)
    got = s.logits()
    at = (0, 255, 256, 2000, 3839, 3840)
    rows = [s.kv(1, p) for p in at]
    s.rewind(0)
    for t in prompt[:-1]:
        s.step_no_output(int(t))
    s.step_greedy(int(prompt[-1]))
    assert rel_l2(got, s.logits()) < 2e-4
    for p, kv in zip(at, rows):
        for a, b in zip(kv, s.kv(1, p)):
            assert rel_l2(a, b) < 2e-3
    s.close()


# hidden, feed-forward, rows in the pass and the tile and split that the named product takes there
PLANS = [(4096, 2048, 3841, {"gate_up": (256, 256, 1)}), (4096, 1024, 3841, {"gate_up": (256, 256, 2)}),
         (4096, 2048, 257, {"gate_up": (256, 256, 8), "o": (256, 256, 8)}), (4096, 2048, 33, {"gate_up": (64, 128, 16)}),
         (2048, 5632, 513, {"gate_up": (128, 128, 1), "down": (256, 256, 8)}), (2048, 2048, 2049, {"qkv": (128, 128, 1)})]


@pytest.mark.parametrize("ttype", [Q4_K, Q6_K, Q8_0, IQ4_XS, Q3_K], ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("hidden,ffn,rows,plan", PLANS, ids=lambda v: str(v) if isinstance(v, int) else "")
def test_tiles_and_splits_match_the_step_path(hip_ctx, ttype, hidden, ffn, rows, plan):
    """Each tile size with gate and up paired, with and without a split.  The plan is asserted, so that a change
    of the estimate's constants can't drop one unseen.  The bars are as above."""
    print(f"tiles {TYPE_NAMES[ttype]} {hidden}/{ffn} rows {rows}", flush=True)
    heads = hidden // 128
    takes = {"qkv": hip.prompt_tiles([hidden, hidden // 4, hidden // 4], rows, hidden),
             "o": hip.prompt_tiles([hidden], rows, hidden), "gate_up": hip.prompt_tiles([ffn], rows, hidden, True),
             "down": hip.prompt_tiles([hidden], rows, ffn)}
    assert {k: takes[k] for k in plan} == plan
    spec = synth.small_spec(hidden=hidden, ffn=ffn, n_head=heads, n_kv=heads // 4, head_dim=128, default_type=ttype,
                            attn_v_type=ttype, output_type=Q8_0, embd_type=Q8_0, context=rows + 63)
    img = synth.build(spec, seed=31)
    prompt = synth.prompt_tokens(4, rows + 1, spec.vocab)
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate(prompt, 0)
    got = s.logits()
    at = (0, rows // 2, rows - 2, rows - 1)
    kv = [s.kv(1, p) for p in at]
    s.rewind(0)
    for t in prompt[:-1]:
        s.step_no_output(int(t))
    s.step_greedy(int(prompt[-1]))
    assert rel_l2(got, s.logits()) < 2e-4
    for p, row in zip(at, kv):
        for a, b in zip(row, s.kv(1, p)):
            assert rel_l2(a, b) < 2e-3
    s.close()
