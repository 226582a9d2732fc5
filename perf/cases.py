"""The framework's ordinary work as measured cases: decode steps and blocks, prompts, a speculative verify
pass, and the MoE stack, each through the public entry points of zhip.hip.

Shapes are the benchmark configurations of this repository (TinyLlama-, Llama-3.1-8B- and Qwen3-8B-shaped
models, the 256-expert MoE stack) and the small shapes of its prompt tests; a case keeps a few of a model's
layers, so that many inputs can be made quickly.  Weights are random codes with the scales that give
N(0, 0.02)-like values.  The output head holds the embedding rows moved by one token, so that a model is as
sure of its next token as a trained one is, and greedy streams don't hang on last bits.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ziggy-llm_amd")
if os.path.isdir(os.path.join(os.getcwd(), "ziggy-llm_amd")):
    _PKG = os.path.join(os.getcwd(), "ziggy-llm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from zhip import gguf, hip, synth  # noqa: E402
from zhip.gguf import F32, IQ4_XS, Q3_K, Q4_K, Q6_K, Q8_0  # noqa: E402

DEV = "cuda"


# ---- models ----

def _spec(model, layers):
    if model == "tinyllama":
        s = synth.tinyllama_spec()
    elif model == "llama8b":
        s = synth.llama8b_spec()
    elif model == "qwen3_8b":
        s = synth.qwen3_8b_spec()
    elif model == "small_q8":  # reductions of an odd number of 256-value chunks
        s = synth.small_spec(hidden=768, ffn=1280, n_head=6, n_kv=2, head_dim=128, default_type=Q8_0,
                             attn_v_type=Q8_0, output_type=Q8_0, embd_type=Q8_0)
    elif model == "small_hd96":
        s = synth.small_spec(hidden=768, ffn=1024, n_head=8, n_kv=2, head_dim=96)
    else:
        raise ValueError(model)
    s.n_layers = layers
    # every second layer's down projection in Q6_K, as in the 32-layer mix
    s.down_q6k_layers = set() if s.default_type == Q8_0 else {i for i in range(layers) if i % 2 == 0}
    # the head is the embedding's rows, so both have the head's format
    s.embd_type = s.output_type
    return s


# ---- random weights in the GGUF block formats, on the GPU ----

def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device=DEV, dtype=torch.uint8)


def _ints(g, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.int32)


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _spread(g, n, base):
    """Per-block scales around `base`."""
    return base * (0.75 + 0.5 * torch.rand(n, generator=g, device=DEV))


def _signed_scales(g, n, k):
    """6-bit scales (stored + 32) of both signs, away from zero."""
    s = _ints(g, 12, 32, n, k)
    return torch.where(_ints(g, 0, 2, n, k) > 0, s, -s) + 32


def _random_matrix(g, ttype, rows, cols, std):
    """[rows, row bytes] uint8: random codes, scales for values of standard deviation `std`."""
    if ttype == F32:
        return (torch.randn(rows, cols, generator=g, device=DEV) * std).view(torch.uint8).reshape(rows, 4 * cols)
    n = rows * cols // gguf.BLOCK[ttype][0]
    if ttype == Q8_0:
        q = _ints(g, -127, 128, n, 32).to(torch.int8).view(torch.uint8)
        b = torch.cat([_f16_bytes(_spread(g, n, std / 73.3)), q], 1)
    elif ttype == Q4_K:
        sc = _ints(g, 24, 64, n, 8)
        mn = (sc + _ints(g, -3, 4, n, 8)).clamp(0, 63)
        d = _spread(g, n, std / (44 * 4.61))
        lo, hi = slice(0, 4), slice(4, 8)
        scales = torch.cat([sc[:, lo] | (sc[:, hi] >> 4 << 6), mn[:, lo] | (mn[:, hi] >> 4 << 6),
                            (sc[:, hi] & 15) | ((mn[:, hi] & 15) << 4)], 1).to(torch.uint8)
        b = torch.cat([_f16_bytes(d), _f16_bytes(7.5 * d), scales, _bytes(g, n, 128)], 1)
    elif ttype == Q6_K:
        s = _ints(g, 40, 128, n, 16)
        s = torch.where(_ints(g, 0, 2, n, 16) > 0, s, -s).to(torch.int8).view(torch.uint8)
        b = torch.cat([_bytes(g, n, 192), s, _f16_bytes(_spread(g, n, std / (86 * 18.5)))], 1)
    elif ttype == IQ4_XS:
        ls = _signed_scales(g, n, 8)
        hi = sum((ls[:, i] >> 4) << (2 * i) for i in range(8))
        sh = torch.stack([hi & 255, hi >> 8], 1).to(torch.uint8)
        sl = ((ls[:, 0::2] & 15) | ((ls[:, 1::2] & 15) << 4)).to(torch.uint8)
        b = torch.cat([_f16_bytes(_spread(g, n, std / (22 * 68.0))), sh, sl, _bytes(g, n, 128)], 1)
    elif ttype == Q3_K:
        ls = _signed_scales(g, n, 16)
        low = ((ls[:, 0:8] & 15) | ((ls[:, 8:16] & 15) << 4)).to(torch.uint8)
        high = sum(((ls[:, 4 * k:4 * k + 4] >> 4) << (2 * k)) for k in range(4)).to(torch.uint8)
        b = torch.cat([_bytes(g, n, 96), low, high, _f16_bytes(_spread(g, n, std / (22 * 2.35)))], 1)
    else:
        raise ValueError(ttype)
    return b.reshape(rows, -1).contiguous()


_IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _values(b, ttype, cols):
    """The matrix of uint8 rows `b` in 64 bits (the GGUF formats' definitions)."""
    rows = b.shape[0]
    if ttype == F32:
        return b.reshape(rows, cols, 4).contiguous().view(torch.float32).reshape(rows, cols).double()
    b = b.reshape(-1, gguf.BLOCK[ttype][1])
    n = b.shape[0]

    def f16(o):
        return b[:, o:o + 2].contiguous().view(torch.float16).double()

    if ttype == Q8_0:
        w = f16(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif ttype == Q4_K:
        s = b[:, 4:16].int()
        lo, mid, top = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (top & 15) | (lo >> 6 << 4)], 1)
        mn = torch.cat([mid & 63, (top >> 4) | (mid >> 6 << 4)], 1)
        q = b[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
        w = (f16(0) * sc)[:, :, None] * q - (f16(2) * mn)[:, :, None]
    elif ttype == Q6_K:
        ql, qh = b[:, :128].reshape(n, 2, 1, 64).int(), b[:, 128:192].reshape(n, 2, 1, 32).int()
        low = torch.cat([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32)
        high = torch.cat([(qh >> (2 * k)) & 3 for k in range(4)], 2)
        q = (low | (high << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * f16(208)
        w = sc[:, :, None] * q.reshape(n, 16, 16).double()
    elif ttype == IQ4_XS:
        sh = b[:, 2].int() | (b[:, 3].int() << 8)
        sl = b[:, 4:8].int()
        low = torch.stack([sl & 15, sl >> 4], 2).reshape(n, 8)
        high = torch.stack([(sh >> (2 * k)) & 3 for k in range(8)], 1)
        dl = f16(0) * ((low | (high << 4)) - 32)
        q = b[:, 8:].reshape(n, 8, 1, 16)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).long()
        w = dl[:, :, None] * torch.tensor(_IQ4, device=b.device, dtype=torch.float64)[q]
    elif ttype == Q3_K:
        hm, qs = b[:, :32].reshape(n, 1, 1, 32).int(), b[:, 32:96].reshape(n, 2, 1, 32).int()
        low2 = torch.cat([(qs >> (2 * k)) & 3 for k in range(4)], 2)
        bit = torch.cat([(hm >> k) & 1 for k in range(8)], 2).reshape(n, 2, 4, 32)
        q = low2 + 4 * bit - 4
        r = b[:, 96:108].int()
        low = torch.cat([r[:, 0:8] & 15, r[:, 0:8] >> 4], 1)
        high = torch.cat([(r[:, 8:12] >> (2 * k)) & 3 for k in range(4)], 1)
        w = (f16(108) * ((low | (high << 4)) - 32))[:, :, None] * q.reshape(n, 16, 16).double()
    else:
        raise ValueError(ttype)
    return w.reshape(rows, cols)


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed & 0x7FFFFFFF)


# ---- dense models ----

def _weights(spec, seed):
    """{tensor name: (uint8 rows, type, cols)} on the GPU."""
    g = _generator(seed)
    got = {}
    for t in spec.tensors():
        if t.name == "output.weight":
            # next-token head: row t + 1 is the embedding of t at an eighth of its size
            e, ttype, cols = got["token_embd.weight"]
            o = e.roll(1, 0).reshape(-1, gguf.BLOCK[ttype][1]).clone()
            at = 208 if ttype == Q6_K else 0
            o[:, at:at + 2] = (o[:, at:at + 2].contiguous().view(torch.float16) / 8).view(torch.uint8)
            m = o.reshape(e.shape)
        elif "norm" in t.name:
            m = (0.75 + 0.5 * torch.rand(t.row_len, generator=g, device=DEV)).view(torch.uint8).reshape(1, -1)
        else:
            m = _random_matrix(g, t.ttype, t.rows, t.row_len, 1.0 if t.name == "token_embd.weight" else 0.02)
        got[t.name] = (m, t.ttype, t.row_len)
    return got


_context = None


def _ctx():
    global _context
    if _context is None:
        _context = hip.Context(0)
    return _context


def _session(spec, weights, context):
    img = gguf.layout([m for m in spec.metadata() if not m[0].startswith("tokenizer")], spec.tensors())
    for name, (m, _, _) in weights.items():
        torch.from_numpy(img.tensor_view(name)).copy_(m.reshape(-1))
    return hip.Session(_ctx(), img, context=context)


def _tokens(case, seed):
    """The tokens the case feeds: those before the call, and the call's own."""
    rng = np.random.default_rng(seed)
    vocab = _spec(case["model"], case["layers"]).vocab
    past = rng.integers(3, vocab, case.get("context", 0)).astype(np.uint32)
    own = rng.integers(3, vocab, case.get("prompt", 1)).astype(np.uint32)
    if case["kind"] == "verify":  # drafts as a good draft model gives them: the model's own next tokens
        own = ((own[:1].astype(np.int64) + np.arange(case["drafts"] + 1)) % vocab).astype(np.uint32)
    return past, own


def _input_row(case, seed):
    """A hidden state in the middle of a model."""
    h = _spec(case["model"], case["layers"]).hidden
    return np.random.default_rng(seed + 1).standard_normal(h).astype(np.float32)


class _Exact:
    """The model in 64 bits: RMSNorm, GQA attention with RoPE over a binary16 cache, SwiGLU."""

    def __init__(self, spec, weights):
        self.s, self.w, self.kept = spec, weights, {}
        self.kv = [[None, None] for _ in range(spec.n_layers)]

    def mat(self, name):
        if name not in self.kept:
            self.kept[name] = _values(*self.w[name])
        return self.kept[name]

    def embed(self, tokens):
        m, ttype, cols = self.w["token_embd.weight"]
        return _values(m[torch.from_numpy(tokens.astype(np.int64)).to(m.device)], ttype, cols)

    def norm(self, x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.s.eps) * self.mat(name)[0]

    def rope(self, x, pos):
        hd = self.s.head_dim
        # base^(2i/n) and the angle are binary32 in the model's definition
        den = torch.tensor([self.s.rope_theta], dtype=torch.float32) ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd)
        a = (pos.float()[:, None] / den.to(pos.device)[None]).double()[:, None, :]
        c, s = torch.cos(a), torch.sin(a)
        y = torch.empty_like(x)
        if self.s.arch == "qwen3":
            u, v, i, j = x[..., :hd // 2], x[..., hd // 2:], slice(0, hd // 2), slice(hd // 2, hd)
        else:
            u, v, i, j = x[..., 0::2], x[..., 1::2], slice(0, hd, 2), slice(1, hd, 2)
        y[..., i], y[..., j] = u * c - v * s, u * s + v * c
        return y

    def attention(self, l, x, pos0):
        s, p, n = self.s, "blk.%d." % l, x.shape[0]
        pos = torch.arange(pos0, pos0 + n, device=x.device)
        y = self.norm(x, p + "attn_norm.weight")
        q = (y @ self.mat(p + "attn_q.weight").T).reshape(n, s.n_head, s.head_dim)
        k = (y @ self.mat(p + "attn_k.weight").T).reshape(n, s.n_kv, s.head_dim)
        v = (y @ self.mat(p + "attn_v.weight").T).reshape(n, s.n_kv, s.head_dim)
        if s.qk_norm:
            q, k = self.norm(q, p + "attn_q_norm.weight"), self.norm(k, p + "attn_k_norm.weight")
        q, k = self.rope(q, pos), self.rope(k, pos)
        for i, new in enumerate((k, v)):  # the cache holds binary16
            new, old = new.half().double(), self.kv[l][i]
            self.kv[l][i] = new if old is None else torch.cat([old[:pos0], new])
        kc, vc = self.kv[l]
        out = torch.empty_like(q)
        grp = s.n_head // s.n_kv
        for h in range(s.n_kv):
            for r in range(0, n, 1024):
                e = min(n, r + 1024)
                qq = q[r:e, h * grp:(h + 1) * grp].transpose(0, 1)
                sc = qq @ kc[:pos0 + e, h].T / math.sqrt(s.head_dim)
                late = torch.arange(pos0 + e, device=x.device)[None, :] > pos[r:e, None]
                pr = torch.softmax(sc.masked_fill(late, -math.inf), -1)
                out[r:e, h * grp:(h + 1) * grp] = (pr @ vc[:pos0 + e, h]).transpose(0, 1)
        return x + out.reshape(n, -1) @ self.mat(p + "attn_output.weight").T

    def ffn(self, l, x):
        p = "blk.%d." % l
        y = self.norm(x, p + "ffn_norm.weight")
        a = torch.nn.functional.silu(y @ self.mat(p + "ffn_gate.weight").T) * (y @ self.mat(p + "ffn_up.weight").T)
        return x + a @ self.mat(p + "ffn_down.weight").T

    def feed(self, tokens, pos0):
        x = self.embed(tokens)
        for l in range(self.s.n_layers):
            x = self.ffn(l, self.attention(l, x, pos0))
        return x

    def logits(self, x):
        return self.norm(x, "output_norm.weight") @ self.mat("output.weight").T


# ---- the MoE stack ----

def _moe_spec(layers):
    return synth.moe_config5_spec(layers)


def _moe_weights(spec, seed):
    g = _generator(seed)
    H, E, F, S = spec.hidden, spec.n_experts, spec.expert_ff, spec.shared_ff
    layers = []
    for _ in range(spec.n_layers):
        m = {"ffn_norm": (0.75 + 0.5 * torch.rand(1, H, generator=g, device=DEV)).view(torch.uint8)}
        shapes = {"ffn_norm": (1, H, F32), "router": (E, H, F32), "gate_exps": (E * F, H, IQ4_XS),
                  "up_exps": (E * F, H, IQ4_XS), "down_exps": (E * H, F, IQ4_XS), "gate_shexp": (S, H, Q3_K),
                  "up_shexp": (S, H, Q3_K), "down_shexp": (H, S, Q3_K), "gate_inp_shexp": (1, H, F32)}
        for k, (rows, cols, t) in shapes.items():
            if k not in m:
                m[k] = _random_matrix(g, t, rows, cols, H ** -0.5 if t == F32 else 0.02)
        layers.append({k: (m[k], shapes[k]) for k in shapes})
    return layers


def _moe_rows(spec, weights, rows, seed):
    """Hidden rows that the routers are sure of: each row leans towards eight experts of every layer."""
    g = _generator(seed + 1)
    x = 0.3 * torch.randn(rows, spec.hidden, generator=g, device=DEV)
    lean = 4.0 + 0.5 * torch.arange(spec.top_k, device=DEV)
    for lay in weights:
        r = lay["router"][0].view(torch.float32).reshape(spec.n_experts, spec.hidden)
        pick = torch.rand(rows, spec.n_experts, generator=g, device=DEV).argsort(1)[:, :spec.top_k]
        x += (r[pick] * lean[None, :, None]).sum(1)
    return x.cpu().numpy()


def _moe_exact(spec, weights, rows):
    x = torch.from_numpy(rows).to(DEV).double()
    n, k, E, F, H = x.shape[0], spec.top_k, spec.n_experts, spec.expert_ff, spec.hidden
    sel, wts = [], []
    for lay in weights:
        def mat(name, lo=0, hi=None):
            m, (_, cols, t) = lay[name]
            return _values(m[lo:hi], t, cols)
        y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + spec.eps) * mat("ffn_norm")[0]
        p = torch.softmax(y @ mat("router").T, -1)
        w, ids = p.topk(k, -1)
        w = w / w.sum(-1, keepdim=True)
        out = torch.zeros_like(x)
        used = torch.unique(ids).tolist()
        for e in used:
            row, slot = torch.nonzero(ids == e, as_tuple=True)
            u = y[row]
            a = torch.nn.functional.silu(u @ mat("gate_exps", e * F, e * F + F).T) * (u @ mat("up_exps", e * F, e * F + F).T)
            out[row] += w[row, slot][:, None] * (a @ mat("down_exps", e * H, e * H + H).T)
        a = torch.nn.functional.silu(y @ mat("gate_shexp").T) * (y @ mat("up_shexp").T)
        x = x + out + torch.sigmoid(y @ mat("gate_inp_shexp").T) * (a @ mat("down_shexp").T)
        sel.append(ids)
        wts.append(w)
    return x, torch.stack(sel, 1), torch.stack(wts, 1)


# ---- the cases ----

def listed():
    return [
        # one small layer through the per-layer calls (hidden state in, hidden state out), as a host that
        # drives the layers itself makes them: launches and latency
        {"name": "block_tiny", "kind": "block", "model": "tinyllama", "layers": 1, "context": 127},
        # the same for a layer of an 8B model at 4k context
        {"name": "block_llama_4k", "kind": "block", "model": "llama8b", "layers": 1, "context": 4099},
        # a short chat turn of a whole small model: prompt and 32 tokens
        {"name": "chat_tiny", "kind": "generate", "model": "tinyllama", "layers": 22, "context": 0, "prompt": 33,
         "steps": 32},
        # ordinary decode at 4k context, Q4_K_M weights
        {"name": "decode_llama_4k", "kind": "generate", "model": "llama8b", "layers": 4, "context": 4096,
         "prompt": 1, "steps": 16},
        # long-context decode, Q8_0 weights and per-head norms
        {"name": "decode_qwen3_16k", "kind": "generate", "model": "qwen3_8b", "layers": 3, "context": 16384,
         "prompt": 1, "steps": 8},
        # one sampled step: the 128256-row head, the shortlist and the logits
        {"name": "sample_llama", "kind": "shortlist", "model": "llama8b", "layers": 1, "context": 611, "count": 40},
        # a short question to an 8B model: time to the first token
        {"name": "prompt_llama_77", "kind": "generate", "model": "llama8b", "layers": 4, "context": 0, "prompt": 77,
         "steps": 1},
        # a long prompt
        {"name": "prompt_llama_4k", "kind": "generate", "model": "llama8b", "layers": 4, "context": 0,
         "prompt": 4096, "steps": 1},
        # the longest prompt, where attention weighs as much as the products
        {"name": "prompt_qwen3_16k", "kind": "generate", "model": "qwen3_8b", "layers": 3, "context": 0,
         "prompt": 16384, "steps": 1},
        # speculative decoding: the pending token and 8 drafts in one pass
        {"name": "verify_qwen3", "kind": "verify", "model": "qwen3_8b", "layers": 4, "context": 2048, "drafts": 8},
        # one token through the MoE layers
        {"name": "moe_token", "kind": "moe", "layers": 4, "rows": 1, "prefill": False},
        # a prompt's rows through the MoE layers
        {"name": "moe_prefill_512", "kind": "moe", "layers": 4, "rows": 512, "prefill": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "decode", "prompt", "prompt", "prompt", "verify", "shortlist", "moe", "moe"])
    if kind == "moe":
        prefill = rng.random() < 0.7
        return {"kind": "moe", "layers": rng.choice([2, 3, 4]), "rows": _log_int(rng, 2, 600) if prefill else 1,
                "prefill": prefill}
    model = rng.choice(["tinyllama", "llama8b", "qwen3_8b", "small_q8", "small_hd96"])
    longest = 12000 if model in ("llama8b", "qwen3_8b") else 6000
    if kind == "block":
        return {"kind": "block", "model": model, "layers": 1, "context": _log_int(rng, 1, longest)}
    if kind == "shortlist":
        return {"kind": "shortlist", "model": model, "layers": 1, "context": _log_int(rng, 1, 3000),
                "count": rng.randint(1, 64)}
    layers = rng.choice([2, 3])
    if kind == "verify":
        return {"kind": "verify", "model": model, "layers": layers, "context": _log_int(rng, 1, 6000),
                "drafts": rng.randint(1, 15)}
    if kind == "decode":
        return {"kind": "generate", "model": model, "layers": layers, "context": _log_int(rng, 1, longest),
                "prompt": 1, "steps": rng.randint(2, 12)}
    # a prompt, at the start of a conversation or after earlier turns
    return {"kind": "generate", "model": model, "layers": layers,
            "context": 0 if rng.random() < 0.6 else _log_int(rng, 5, 4000), "prompt": _log_int(rng, 2, longest),
            "steps": 1}


def _kept_rows(case):
    """The prompt rows whose last-layer cache entries a case returns: a third of the way, and the last but one."""
    n = case["prompt"]
    return (n // 3, n - 2) if n > 1 else ()


def prepare(case, seed):
    if case["kind"] == "moe":
        spec = _moe_spec(case["layers"])
        w = _moe_weights(spec, seed)
        layers = [{k: (m.reshape(-1).cpu().numpy(), rows, cols, t) for k, (m, (rows, cols, t)) in lay.items()}
                  for lay in w]
        rows = _moe_rows(spec, w, case["rows"], seed)
        return {"case": case, "stack": hip.MoeStack(_ctx(), synth.moe_desc(spec), layers), "rows": rows}
    spec = _spec(case["model"], case["layers"])
    past, own = _tokens(case, seed)
    room = len(past) + len(own) + case.get("steps", 0) + 1
    s = _session(spec, _weights(spec, seed), room)
    if len(past):
        s.generate(past, 0)
    state = {"case": case, "session": s, "past": len(past), "own": own}
    if case["kind"] == "block":
        state["row"] = _input_row(case, seed)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "moe":
        if case["prefill"]:
            return state["stack"].prefill(state["rows"])
        return state["stack"].forward(state["rows"][0])
    s, past, own = state["session"], state["past"], state["own"]
    if case["kind"] == "block":
        s.begin_token(state["row"])
        s.run_attention_block(0, past)
        s.run_ffn_block(0)
        return s.hidden()
    s.rewind(past)  # the same turn again
    if case["kind"] == "generate":
        tokens, _ = s.generate(own, case["steps"])
        return (tokens, s.logits()) + tuple(s.kv(case["layers"] - 1, past + i) for i in _kept_rows(case))
    if case["kind"] == "shortlist":
        ids, scores = s.step_shortlist(int(own[0]), case["count"])
        return ids, scores, s.logits()
    predicted, count = s.verify(int(own[0]), own[1:])
    # the last layer's cache row of the last draft, which the next pass reads
    return predicted, count, s.kv(case["layers"] - 1, past + len(own) - 1)


def exact(case, seed):
    if case["kind"] == "moe":
        spec = _moe_spec(case["layers"])
        w = _moe_weights(spec, seed)
        x, sel, wts = _moe_exact(spec, w, _moe_rows(spec, w, case["rows"], seed))
        return (x, None, wts) if case["prefill"] else (x[0], None, wts[0])
    spec = _spec(case["model"], case["layers"])
    past, own = _tokens(case, seed)
    m = _Exact(spec, _weights(spec, seed))
    if case["kind"] == "block":
        for l in range(spec.n_layers):
            m.attention(l, m.embed(past), 0)
        x = torch.from_numpy(_input_row(case, seed)).to(DEV).double()[None]
        return m.ffn(0, m.attention(0, x, len(past)))[0]
    if len(past):
        m.feed(past, 0)
    if case["kind"] == "shortlist":
        lg = m.logits(m.feed(own, len(past))[-1:])[0]
        return None, lg.topk(case["count"]).values, lg
    if case["kind"] == "verify":
        m.feed(own, len(past))
        return None, None, (m.kv[-1][0][-1].reshape(-1), m.kv[-1][1][-1].reshape(-1))
    pos = len(past) + len(own)
    lg = m.logits(m.feed(own, len(past))[-1:])[0]
    for _ in range(case["steps"]):
        lg = m.logits(m.feed(np.array([int(lg.argmax())], np.uint32), pos)[-1:])[0]
        pos += 1
    rows = tuple(tuple(c[len(past) + i].reshape(-1) for c in m.kv[-1]) for i in _kept_rows(case))
    return (None, lg) + rows


def work(case):
    """Weights and cache rows read and written once per pass over them, multiply-adds counted twice."""
    if case["kind"] == "moe":
        spec, n = _moe_spec(case["layers"]), case["rows"]
        one, most = spec.weight_bytes_per_token(), spec.weight_bytes_all()
        # the routed experts that n rows reach when each takes top_k of all
        part = 1 - (1 - spec.top_k / spec.n_experts) ** n
        per_expert = (most - one) / (spec.n_experts - spec.top_k)
        return {"bytes": one + per_expert * (part * spec.n_experts - spec.top_k) + 8 * n * spec.hidden,
                "flops": n * spec.flops_per_token()}
    spec = _spec(case["model"], case["layers"])
    L, H, Q, KV = spec.n_layers, spec.hidden, spec.n_head * spec.head_dim, spec.n_kv * spec.head_dim
    layer_bytes = sum(t.nbytes for t in spec.tensors() if t.name.startswith("blk."))
    head = [t for t in spec.tensors() if t.name == "output.weight"][0]
    past = case.get("context", 0)

    def rows(n, at, last_only):
        """n rows from position `at` through the layers: (flops, cache bytes)."""
        seen = n * at + n * (n + 1) // 2
        f = L * (2 * n * spec.matmul_params_per_layer() + 4 * Q * seen)
        if last_only:  # what comes after the last layer's cache rows is needed for the last row alone
            drop = n - 1
            f -= 2 * drop * (spec.matmul_params_per_layer() - 2 * H * KV) + 4 * Q * (seen - at - n)
        return f, L * 4 * KV * (at + n)

    if case["kind"] == "block":
        f, b = rows(1, past, False)
        return {"bytes": layer_bytes + b + 8 * H, "flops": f}
    if case["kind"] == "shortlist":
        f, b = rows(1, past, False)
        return {"bytes": layer_bytes + head.nbytes + b, "flops": f + 2 * H * spec.vocab}
    if case["kind"] == "verify":
        n = case["drafts"] + 1
        f, b = rows(n, past, False)
        return {"bytes": layer_bytes + head.nbytes + b, "flops": f + 2 * n * H * spec.vocab}
    f, b = rows(case["prompt"], past, True)
    total = {"bytes": layer_bytes + head.nbytes + b, "flops": f + 2 * H * spec.vocab}
    for i in range(case["steps"]):
        f, b = rows(1, past + case["prompt"] + i, False)
        total["bytes"] += layer_bytes + head.nbytes + b
        total["flops"] += f + 2 * H * spec.vocab
    return total


def tolerance(case):
    # About four times the distance to exact() over listed and drawn cases.  Activations are binary32; a last
    # bit can move a cache entry by one binary16 step (up to 1e-3 of it), and later layers carry that on.
    if case["kind"] == "moe":
        return {"rel": 1e-5, "max": 5e-4, "differ": 0.002}
    if case["kind"] == "block":
        return {"rel": 5e-5, "max": 5e-4}
    return {"rel": 1.2e-3, "max": 1e-2, "differ": 0.002}
