"""A prompt's passes under the switches that change their products or their length.

The switches are read once per process, so each run is a child process: it feeds the prompts one after the
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

MODELS = {
    "q4km-g2": dict(down_q6k_layers=[1], context=512),
}


def _model(name):
    from zhip import synth
    spec = synth.small_spec(**MODELS[name])
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


if __name__ == "__main__":
    sys.path[:0] = [REPO, os.path.join(REPO, "ziggy-llm_amd")]
    _child(*json.loads(sys.argv[1]))
