"""A prompt's passes: where one ends and the next begins, models that mix products, and the switches that
change their products or their length.

The switches are read once per process, so such a run is a child process: it feeds the prompts one after the
other and leaves the logits and the K/V rows of chosen positions.  Logits within 1e-4 relative L2 of the
oracle's token-by-token prompt and K/V rows within 1e-3 (one binary16 step), as in test_gpu_prefill.py.
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [p for p in (REPO, os.path.join(REPO, "ziggy-llm_amd")) if p not in sys.path]

from zhip.gguf import F32, Q4_K, Q8_0  # noqa: E402

MODELS = {
    "q4km-g2": dict(down_q6k_layers=[1], context=640),
    # matrices that the prompt products don't take, so passes of 256 rows: a gate of F32 values beside an up of
    # Q4_K, F32 queries, keys and values, and a down projection whose 320 values are no multiple of 256
    "f32-gate": dict(down_q6k_layers=[0], context=700),
    "f32-qkv": dict(context=700),
    "q8-ffn-320": dict(ffn=320, n_head=4, n_kv=1, default_type=Q8_0, attn_v_type=Q8_0, output_type=Q8_0,
                       embd_type=Q8_0, context=700),
}
IN_F32 = {"f32-gate": ("ffn_gate.weight",), "f32-qkv": ("attn_q.weight", "attn_k.weight", "attn_v.weight")}


def _model(name):
    from zhip import synth
    spec = synth.small_spec(**MODELS[name])
    tensors = spec.tensors()
    for t in tensors:
        if t.name.endswith(IN_F32.get(name, ())):
            t.ttype = F32
    spec.tensors = lambda: tensors
    return spec, synth.build(spec, seed=71)


def _turns(spec, lengths):
    from zhip import synth
    return [synth.prompt_tokens(72 + i, n, spec.vocab) for i, n in enumerate(lengths)]


def _child(out, name, lengths, positions):
    from zhip import hip
    spec, img = _model(name)
    ctx = hip.Context(0)
    s = hip.Session(ctx, img, context=spec.context)
    for t in _turns(spec, lengths):
        s.generate(t, 0)
    rows = [[s.kv(layer, p) for p in positions] for layer in range(spec.n_layers)]
    np.savez(out, logits=s.logits(), rows=np.array(rows))
    s.close()
    ctx.close()


def passes(tmp_path, name, lengths, positions, **env):
    out = str(tmp_path / "rows.npz")
    args = json.dumps([out, name, lengths, positions])
    print(f"prompt passes {name} {lengths} {env}", flush=True)
    subprocess.run([sys.executable, os.path.abspath(__file__), args], check=True, timeout=100,
                   env={**os.environ, **env})
    z = np.load(out)
    return z["logits"], z["rows"]


def rel_l2(a, b):
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def check(name, lengths, positions, logits, rows):
    from oracle import zo
    spec, img = _model(name)
    o = zo.Session(zo.Model(img.buf), context=spec.context, kv_f16=True)
    tokens = np.concatenate(_turns(spec, lengths))
    for t in tokens[:-1]:
        o.step_no_output(int(t))
    assert rel_l2(logits, o.step(int(tokens[-1]))) < 1e-4
    for layer in range(spec.n_layers):
        for i, p in enumerate(positions):
            for a, b in zip(rows[layer][i], o.kv(layer, p)):
                assert rel_l2(a, b) < 1e-3, (layer, p)


@pytest.mark.gpu
def test_qgemm_switch_reaches_the_prompt_products(tmp_path):
    """ZIGGY_HIP_QGEMM=0 runs a prompt's products on the decoding kernel (and ZIGGY_HIP_VERIFY_SWIGLU=fused its
    gate and up as one): other last bits, the same bars."""
    at = [0, 33, 64, 288]
    default = passes(tmp_path, "q4km-g2", [290], at)
    off = passes(tmp_path, "q4km-g2", [290], at, ZIGGY_HIP_QGEMM="0")
    fused = passes(tmp_path, "q4km-g2", [290], at, ZIGGY_HIP_QGEMM="0", ZIGGY_HIP_VERIFY_SWIGLU="fused")
    for got in (default, off, fused):
        check("q4km-g2", [290], at, *got)
    assert (default[1] != off[1]).any()


# rows fed in passes of 64: four and a ragged one, one and a last one of 5 rows (the verify pass's products),
# and of exactly 64
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [299, 69, 261, 128])
def test_pass_boundaries(tmp_path, rows):
    at = sorted({p for p in (0, 63, 64, 127, 128, 255, 256, rows - 6, rows - 1) if p < rows})
    got = passes(tmp_path, "q4km-g2", [rows + 1], at, ZIGGY_HIP_PREFILL_CHUNK="64")
    check("q4km-g2", [rows + 1], at, *got)


# turns of one session: passes of 256 rows and of the rest; a longer prompt after a shorter one, whose buffers
# grow in between for the models that take long passes; and the same rows again
@pytest.mark.gpu
@pytest.mark.parametrize("name,turns", [("f32-gate", [600]), ("f32-gate", [30, 523]), ("f32-qkv", [290]),
                                        ("q8-ffn-320", [600]), ("q8-ffn-320", [262, 300]),
                                        ("q4km-g2", [20, 300, 130]), ("q4km-g2", [258, 5, 240])])
def test_turns_of_one_session(hip_ctx, name, turns):
    from zhip import hip
    print(f"turns {name} {turns}", flush=True)
    spec, img = _model(name)
    s = hip.Session(hip_ctx, img, context=spec.context)
    n = sum(turns)
    at = sorted({p for p in (0, 17, 255, 256, *(sum(turns[:i]) for i in range(1, len(turns))), 511, 512, n - 2)
                 if p < n - 1})
    runs = []
    for _ in range(2):
        for t in _turns(spec, turns):
            s.generate(t, 0)
        runs.append((s.logits(), np.array([[s.kv(layer, p) for p in at] for layer in range(spec.n_layers)])))
        s.rewind(0)
    check(name, turns, at, *runs[0])
    assert (runs[0][1] == runs[1][1]).all()  # the passes' sums have a fixed order
    s.close()


# a second pass behind one of 4096 rows: of 7 rows, and of 300
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [4103, 4396])
def test_longest_pass_and_the_next(hip_ctx, rows):
    """Against the same prompt token by token through the decode step, which has the oracle's bars of 1e-4 and
    1e-3: twice those."""
    from zhip import hip, synth
    print(f"longest pass, {rows} rows", flush=True)
    spec = synth.small_spec(default_type=Q4_K, context=4480)
    img = synth.build(spec, seed=73)
    prompt = synth.prompt_tokens(74, rows + 1, spec.vocab)
    s = hip.Session(hip_ctx, img, context=spec.context)
    s.generate(prompt, 0)
    got, at = s.logits(), (0, 4095, 4096, 4102, rows - 1)
    kv = [s.kv(1, p) for p in at]
    s.rewind(0)
    for t in prompt[:-1]:
        s.step_no_output(int(t))
    s.step_greedy(int(prompt[-1]))
    assert rel_l2(got, s.logits()) < 2e-4
    for p, rows_p in zip(at, kv):
        for a, b in zip(rows_p, s.kv(1, p)):
            assert rel_l2(a, b) < 2e-3, p
    s.close()


if __name__ == "__main__":
    _child(*json.loads(sys.argv[1]))
