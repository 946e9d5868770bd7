"""Performance cases: the calls a serving program makes, at the Qwen3-30B-A3B
shape (dim 2048, 128 experts, top-8, expert width 768; attention 32/4 heads
of 128; vocabulary 151936), through the library's public entry points.

kinds
  decode  mia_moe_decode: one token through L MoE layers, host x in and out
          (a decode step's FFN path: one layer is the smallest call there is,
          48 layers a whole model's)
  layer   mia_moe_layer_dev: one MoE layer over T tokens resident in HBM (small
          batches of sequences, prompt chunks of any length, long prompts,
          and a router skewed by a per-expert bias)
  stack   mia_moe_stack_graph: batched decode, T sequences through L layers,
          replayed as one graph from the server's fixed x buffer
  attn    mhip_attention_batch: one layer's attention of a prompt chunk of n
          tokens at position pos of its context
  step    mia_gpu_model_step: a whole model's decode step at position pos of a
          conversation, logits out
  prompt  mia_gpu_model_prefill + mia_gpu_model_step: a whole prompt of n
          tokens, logits of its last token out
  sample  mhip_sample: the token sampler on device logits

Handles (weights, KV prefix) are opened once and kept, as a program keeps
them; the inputs come from the seed. Calls that work in place get their input
by a device copy into the program's x buffer first. Every path is specified
bit for bit (the reference's operation order), so outputs compare exactly.
"""
import ctypes
import math

import numpy as np
import torch

import motoria_amd as M
from motoria_amd import workloads as W

D, E, K, EH = 2048, 128, 8, 768
NH, NKV, HD = 32, 4, 128
QD, KVD = NH * HD, NKV * HD
VOCAB = 151936
EPS = 1e-6
ROPE_THETA = 1e6
LAYERS = 48
BLOB = 3 * EH * D // 32 * 36          # Q8_0 bytes of one expert
MAX_T = 4096                          # tokens of the layer handle
CTX = 4096                            # context of the model handle
TOP = 4                               # layers of the layer handle
SIGMA = 0.02

_keep = {}


def listed():
    return [
        # one token, one layer: the smallest call of the engine's FFN entry
        {"name": "decode 1 layer", "kind": "decode", "layers": 1},
        # one token through every layer: batch-1 generation
        {"name": "decode 48 layers", "kind": "decode", "layers": LAYERS},
        # a few sequences decoding together
        {"name": "layer 13 tokens", "kind": "layer", "tokens": 13, "skew": False},
        # a full server batch decoding
        {"name": "stack 64 tokens", "kind": "stack", "tokens": 64, "layers": TOP},
        # a short prompt, of no special length
        {"name": "layer 203 tokens", "kind": "layer", "tokens": 203, "skew": False},
        # a prompt chunk
        {"name": "layer 512 tokens", "kind": "layer", "tokens": 512, "skew": False},
        # uneven expert load
        {"name": "layer 2048 tokens skewed", "kind": "layer", "tokens": 2048, "skew": True},
        # the largest layer call
        {"name": "layer 4096 tokens", "kind": "layer", "tokens": 4096, "skew": False},
        # a prompt chunk's attention behind a context
        {"name": "attention chunk", "kind": "attn", "tokens": 777, "pos": 1200},
        # generation deep in a conversation
        {"name": "model step", "kind": "step", "pos": 2500},
        # a document as the prompt
        {"name": "model prompt", "kind": "prompt", "tokens": 1400},
        # drawing the token (the settings of the repository's sampler benchmark)
        {"name": "sample", "kind": "sample", "temperature": 0.8, "top_p": 0.95},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "layer", "layer", "layer", "layer", "stack", "attn", "step",
                       "prompt", "sample"])
    if kind == "decode":
        return {"kind": kind, "layers": _log(rng, 2, LAYERS - 1)}
    if kind == "layer":
        t = _log(rng, 1, MAX_T)
        return {"kind": kind, "tokens": t, "skew": rng.random() < 0.25}
    if kind == "stack":
        return {"kind": kind, "tokens": _log(rng, 2, 256), "layers": rng.randint(2, TOP)}
    if kind == "attn":
        return {"kind": kind, "tokens": _log(rng, 2, 1024), "pos": rng.choice([0, _log(rng, 16, 2000)])}
    if kind == "step":
        return {"kind": kind, "pos": _log(rng, 16, CTX - 1)}
    if kind == "prompt":
        return {"kind": kind, "tokens": _log(rng, 16, 1400)}
    return {"kind": kind, "temperature": rng.choice([0.6, 0.7, 0.8, 1.0]),
            "top_p": round(rng.uniform(0.8, 1.0), 2)}


# ---- weights and inputs -------------------------------------------------------------

def _gen(*key):
    g = torch.Generator("cuda")
    g.manual_seed(sum((int(k) + 1) * p for k, p in zip(key, (1000003, 7919, 104729, 15485863))))
    return g


def _q8(x):
    """Q8_0 of rows of 32-blocks in float32: (codes int8, scales)."""
    b = x.reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    v = b * inv
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    return q.to(torch.int8), d


def _blocks(x):
    """The 36-byte Q8_0 blocks of x (scale, 32 codes), as bytes."""
    q, d = _q8(x)
    return torch.cat([d.contiguous().view(torch.uint8).reshape(-1, 4), q.view(torch.uint8)], 1).reshape(-1)


def _dequant(x):
    q, d = _q8(x)
    return (q.double() * d.double()).reshape(x.shape)


def _matrix(rows, cols, *key):
    return torch.randn(rows, cols, device="cuda", generator=_gen(*key)) * SIGMA


def _expert(layer, e):
    """gate, up [EH][D] and down [D][EH] of an expert, before quantization."""
    k = 3 * (layer * E + e)
    return _matrix(EH, D, 11, k), _matrix(EH, D, 11, k + 1), _matrix(D, EH, 11, k + 2)


def _dense(layer):
    """ffn_norm [D] and router [E][D]."""
    norm = 1.0 + 0.1 * torch.randn(D, device="cuda", generator=_gen(12, layer))
    return norm, _matrix(E, D, 13, layer)


def _moe_layers():
    """A handle with TOP layers of known weights (the layer and stack cases)."""
    if "layers" not in _keep:
        m = M.Moe(TOP, MAX_T)
        for l in range(TOP):
            norm, router = _dense(l)
            m.set_layer(l, norm.cpu().numpy(), router.cpu().numpy())
            for e in range(E):
                blob = np.zeros(m.blob_bytes, np.uint8)
                for off, w in zip((0, m.off_up, m.off_down), _expert(l, e)):
                    b = _blocks(w).cpu().numpy()
                    blob[off:off + b.size] = b
                m.load_expert(l, e, blob)
        _keep["layers"] = m
        _keep["work"] = torch.empty(MAX_T, D, device="cuda")
        _keep["bias"] = torch.from_numpy(W.zipf_bias(E)).cuda()
    return _keep["layers"]


def _moe_deep():
    """A whole model's MoE layers (36 GB of experts)."""
    if "deep" not in _keep:
        m = M.Moe(LAYERS, 1)
        m.synth(W.WEIGHT_SEED)
        _keep["deep"] = m
    return _keep["deep"]


def _prefix():
    return np.random.default_rng(5).integers(0, VOCAB, CTX).astype(np.int32)


def _model():
    """A whole model and the KV rows of a conversation of CTX tokens."""
    if "model" not in _keep:
        shape = dict(dim=D, n_layers=LAYERS, n_heads=NH, n_kv_heads=NKV, head_dim=HD, vocab=VOCAB,
                     n_experts=E, n_active=K, expert_hidden=EH, norm_topk=1,
                     rope_theta=ROPE_THETA, norm_eps=EPS)
        _keep["model"] = M.GpuModel(None, CTX, synth=(shape, W.WEIGHT_SEED))
        _keep["rows"] = None          # positions whose KV rows are not the conversation's
    return _keep["model"]


def _conversation(pos):
    """The model with the conversation's KV rows below pos."""
    m = _model()
    if _keep["rows"] is None:         # (None: all of them)
        m.prefill(_prefix()[:CTX - 1], 0)
        _keep["rows"] = set()
    for p in sorted(_keep["rows"]):
        if p < pos:
            m.feed(int(_prefix()[p]), p)
    _keep["rows"] = {p for p in _keep["rows"] if p >= pos} | {pos}
    return m


def _gpu():
    if "gpu" not in _keep:
        _keep["gpu"] = M.Gpu()
    return _keep["gpu"]


def _attn_dims():
    return M.AttnDims(D, NH, NKV, HD, EPS)


def _rope(n):
    i = torch.arange(HD // 2, dtype=torch.float64, device="cuda")
    a = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * ROPE_THETA ** (-2.0 * i / HD)
    return torch.stack([a.cos(), a.sin()], -1).contiguous()


def _attn_weights():
    return [_matrix(r, c, 21, k) for k, (r, c) in
            enumerate(((QD, D), (KVD, D), (KVD, D), (D, QD)))]


def _x(tokens, seed):
    return torch.randn(tokens, D, device="cuda", generator=_gen(31, seed))


def _kv(rows, seed):
    """Cached keys (normalised, rotated) and values."""
    g = _gen(32, seed)
    k = torch.randn(rows, KVD, device="cuda", generator=g)
    v = torch.randn(rows, KVD, device="cuda", generator=g) * (SIGMA * math.sqrt(D))
    return k, v


def _logits(seed):
    """Logits with a model's spread: a broad body and a few likely tokens."""
    g = _gen(33, seed)
    l = torch.randn(VOCAB, device="cuda", generator=g) * 2.5
    best = torch.randint(0, VOCAB, (40,), device="cuda", generator=g)
    l[best] += 8.0 + 6.0 * torch.rand(40, device="cuda", generator=g)
    return l.contiguous()


# ---- the interface ---------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        m = _moe_layers() if case["layers"] <= TOP else _moe_deep()
        x = np.random.default_rng(seed).standard_normal(D).astype(np.float32)
        return {"kind": kind, "m": m, "x": x, "layers": case["layers"]}
    if kind in ("layer", "stack"):
        return {"kind": kind, "m": _moe_layers(), "x": _x(case["tokens"], seed), "case": case}
    if kind == "attn":
        n, pos = case["tokens"], case["pos"]
        a, g, L = _attn_dims(), _gpu(), M.lib()
        w = [_blocks(t) for t in _attn_weights()]
        s = {"kind": kind, "x": _x(n, seed), "w": w, "a": a, "n": n, "pos": pos, "seq": pos + n}
        s["norm"] = torch.ones(D, device="cuda")
        s["hnorm"] = torch.ones(HD, device="cuda")
        s["rope"] = _rope(pos + n)
        k, v = _kv(pos, seed)
        new = torch.zeros(n, KVD, device="cuda")
        s["kc"], s["vc"] = torch.cat([k, new]).contiguous(), torch.cat([v, new]).contiguous()
        s["out"] = torch.empty_like(s["x"])
        s["scratch"] = torch.zeros(L.mhip_attention_batch_scratch_bytes(ctypes.byref(a), n, pos + n),
                                   dtype=torch.uint8, device="cuda")
        s["pack"] = torch.empty(L.mhip_attention_pack_bytes(ctypes.byref(a)), dtype=torch.uint8,
                                device="cuda")
        torch.cuda.synchronize()
        g.check(L.mhip_attention_pack(g.h, ctypes.byref(a), *[t.data_ptr() for t in w],
                                      s["pack"].data_ptr()), "pack")
        return s
    if kind == "step":
        token = int(np.random.default_rng(seed).integers(0, VOCAB))
        return {"kind": kind, "m": _conversation(case["pos"]), "token": token, "pos": case["pos"]}
    if kind == "prompt":
        tokens = np.random.default_rng(seed).integers(0, VOCAB, case["tokens"]).astype(np.int32)
        m = _model()
        _keep["rows"] = None
        return {"kind": kind, "m": m, "tokens": tokens}
    if kind == "sample":
        l = _logits(seed)
        return {"kind": kind, "logits": l, "case": case, "seed": seed + 1,
                "scratch": torch.empty(M.lib().mhip_sample_scratch_bytes(VOCAB), dtype=torch.uint8,
                                       device="cuda"),
                "token": torch.zeros(1, dtype=torch.int32, device="cuda")}
    raise ValueError(kind)


def run(s):
    kind, L = s["kind"], M.lib()
    if kind == "decode":
        return s["m"].decode(0, s["layers"], s["x"])
    if kind in ("layer", "stack"):
        m, c, x = s["m"], s["case"], s["x"]
        t = c["tokens"]
        work = _keep["work"]
        if L.mhip_d2d(m.gpu, work.data_ptr(), x.data_ptr(), t * D * 4):
            raise RuntimeError("mhip_d2d")
        if kind == "stack":
            m.stack_graph(0, c["layers"], work.data_ptr(), t)
        else:
            m.layer_dev(0, work.data_ptr(), t, _keep["bias"].data_ptr() if c["skew"] else None)
        return work[:t]
    if kind == "attn":
        g, a = _gpu(), s["a"]
        g.check(L.mhip_d2d(g.h, s["out"].data_ptr(), s["x"].data_ptr(), s["n"] * D * 4), "mhip_d2d")
        w = [t.data_ptr() for t in s["w"]]
        g.check(L.mhip_attention_batch(
            g.h, ctypes.byref(a), s["norm"].data_ptr(), *w, s["hnorm"].data_ptr(),
            s["hnorm"].data_ptr(), s["rope"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(),
            s["pos"], s["n"], s["seq"], s["out"].data_ptr(), s["pack"].data_ptr(),
            s["scratch"].data_ptr(), 0), "mhip_attention_batch")
        return s["out"], s["kc"][s["pos"]:], s["vc"][s["pos"]:]
    if kind == "step":
        return s["m"].step(s["token"], s["pos"])
    if kind == "prompt":
        t = s["tokens"]
        s["m"].prefill(t[:-1], 0)
        return s["m"].step(int(t[-1]), len(t) - 1)
    sm = M.sampler(s["case"]["temperature"], s["case"]["top_p"], VOCAB, s["seed"])
    M.sample_dev(_gpu(), sm, s["logits"].data_ptr(), s["scratch"].data_ptr(), s["token"].data_ptr())
    return s["token"]


def _touched(a):
    """Experts that `a` assignments, K a token, reach when spread evenly."""
    return E * (1.0 - (1.0 - K / E) ** (a / K))


def _layer_work(t):
    return (_touched(t * K) * BLOB + E * D * 4 + 2 * t * D * 4,
            t * (K * 3 * EH * D * 2 + E * D * 2))


def _attn_work(n, pos):
    rows = QD + 2 * KVD
    pairs = n * pos + n * (n + 1) // 2
    return ((rows * D + D * QD) // 32 * 36 + 2 * n * D * 4 + 2 * (pos + 2 * n) * KVD * 4,
            2 * n * (rows * D + D * QD) + 4 * pairs * QD)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        b, f = _layer_work(1)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind in ("layer", "stack"):
        b, f = _layer_work(case["tokens"])
        return {"bytes": case.get("layers", 1) * b, "flops": case.get("layers", 1) * f}
    if kind == "attn":
        b, f = _attn_work(case["tokens"], case["pos"])
        return {"bytes": b, "flops": f}
    if kind in ("step", "prompt"):
        n, pos = (1, case["pos"]) if kind == "step" else (case["tokens"], 0)
        (ab, af), (mb, mf) = _attn_work(n, pos), _layer_work(n)
        return {"bytes": LAYERS * (ab + mb) + VOCAB * D // 32 * 36 + VOCAB * 4,
                "flops": LAYERS * (af + mf) + 2 * VOCAB * D}
    return {"bytes": VOCAB * 4, "flops": VOCAB}


def tolerance(case):
    # Every entry point is specified to the bit (the same operations in the
    # same order), and two runs of the same inputs agree to the bit.
    return "exact"


# ---- the same values in 64 bits ------------------------------------------------------------

def _act(x):
    """Q8_0 of activations, as the model defines its products, in 64 bits."""
    b = x.reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127.0
    v = torch.where(d != 0, b / d, torch.zeros_like(b))
    return (torch.sign(v) * torch.floor(v.abs() + 0.5) * d).reshape(x.shape)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _exact_layer(layer, x, bias=None):
    norm, router = _dense(layer)
    xn = _rms(x, norm.double())
    logits = xn @ router.double().T
    if bias is not None:
        logits = logits + bias.double()
    p = torch.softmax(logits, -1)
    w, idx = torch.topk(p, K, dim=-1)
    w = w / w.sum(-1, keepdim=True)
    xq, y = _act(xn), x.clone()
    for e in range(E):
        t, j = torch.nonzero(idx == e, as_tuple=True)
        if not len(t):
            continue
        gate, up, down = (_dequant(m) for m in _expert(layer, e))
        g, u = xq[t] @ gate.T, xq[t] @ up.T
        h = _act(g / (1.0 + torch.exp(-g)) * u)
        y.index_add_(0, t, (h @ down.T) * w[t, j][:, None])
    return y, idx, w


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode" and case["layers"] == 1:
        x = np.random.default_rng(seed).standard_normal(D).astype(np.float32)
        y, idx, w = _exact_layer(0, torch.from_numpy(x).cuda().double()[None])
        return y[0], idx.to(torch.int32), w
    if kind == "layer":
        bias = torch.from_numpy(W.zipf_bias(E)).cuda() if case["skew"] else None
        return _exact_layer(0, _x(case["tokens"], seed).double(), bias)[0]
    if kind == "attn":
        n, pos = case["tokens"], case["pos"]
        x = _x(n, seed).double()
        wq, wk, wv, wo = (_dequant(t) for t in _attn_weights())
        xq = _act(_rms(x, 1.0))
        rope = _rope(pos + n)[pos:]

        def rot(h):
            h = _rms(h, 1.0)
            a, b = h[..., :HD // 2], h[..., HD // 2:]
            c, s = rope[:, None, :, 0], rope[:, None, :, 1]
            return torch.cat([a * c - b * s, a * s + b * c], -1)

        q = rot((xq @ wq.T).reshape(n, NH, HD))
        k = rot((xq @ wk.T).reshape(n, NKV, HD))
        v = (xq @ wv.T).reshape(n, NKV, HD)
        kc, vc = (t.double().reshape(pos, NKV, HD) for t in _kv(pos, seed))
        kk, vv = torch.cat([kc, k]), torch.cat([vc, v])
        seen = torch.arange(pos + n, device="cuda")[None] <= torch.arange(pos, pos + n, device="cuda")[:, None]
        att = torch.empty(n, NH, HD, dtype=torch.float64, device="cuda")
        for h in range(NH):
            s = q[:, h] @ kk[:, h // (NH // NKV)].T / math.sqrt(HD)
            s = s.masked_fill(~seen, float("-inf"))
            att[:, h] = torch.softmax(s, -1) @ vv[:, h // (NH // NKV)]
        return x + _act(att.reshape(n, QD)) @ wo.T, k.reshape(n, KVD), v.reshape(n, KVD)
    return None
