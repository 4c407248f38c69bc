"""What a user of this framework has it do, through its public entry points, for measuring.

The work is a wick session's: attention over the device-resident KV cache for one
token, for a prompt and for a new turn on a kept prefix (DeviceKvCache); the whole
forward and the greedy loop (DeviceModel); one draw (DeviceSampler).  The shapes
are those of the repository's configurations: SmolLM2-135M, the attention of
Qwen2.5-0.5B, Qwen3-0.6B, TinyLlama-1.1B and Llama-3-8B, all in f32.

listed() names the cases, draw() gives more of the same ranges, prepare() / run()
make and do one pass, work() is what a pass cannot do without, exact() the same
result in 64 bits by plain torch.
"""
import math

import numpy as np
import torch

from wick_amd.device_model import DeviceModel
from wick_amd.kv import DeviceKvCache
from wick_amd.model import Config
from wick_amd.sampler import DeviceSampler, SamplerConfig

DEV = "cuda"

# attention of the configurations: query heads, kv heads, head_dim, RoPE theta, QK-norm, biases
SHAPES = {
    "smollm2": (9, 3, 64, 1e4, False, False),
    "qwen2.5": (14, 2, 64, 1e6, False, True),
    "qwen3": (16, 8, 128, 1e6, True, False),
    "tinyllama": (32, 4, 64, 1e4, False, False),
    "llama3": (32, 8, 128, 5e5, False, False),
}

# whole models and stacks of layers: attention shape, hidden, intermediate, layers, vocabulary
MODELS = {
    # SmolLM2-135M entire (tied embeddings)
    "smollm2-135m": ("smollm2", 576, 1536, 30, 49152),
    # two layers of TinyLlama-1.1B's size under an LM head
    "tinyllama-2l": ("tinyllama", 2048, 5632, 2, 32000),
    # one layer of Llama-3-8B's size under an LM head of 32000 rows
    "llama3-1l": ("llama3", 4096, 14336, 1, 32000),
}


def listed():
    return [
        # one decode step's attention over every layer, at the longest context served
        # by the small models: 24 layers x 33.5 MB of keys and values
        dict(name="decode-qwen2.5-32k", kind="decode", shape="qwen2.5", layers=24, t=1, start=32767, prep=False),
        # a decode step of a large model at a long context, raw q/k/v in and the new
        # key appended (4 of its 32 layers)
        dict(name="decode-llama3-64k", kind="decode", shape="llama3", layers=4, t=1, start=65500, prep=True),
        # a prompt's attention in one layer: QK-norm, RoPE, append, causal attention
        dict(name="prompt-qwen3-512", kind="prompt", shape="qwen3", layers=1, t=512, start=0, prep=True),
        dict(name="prompt-qwen3-2048", kind="prompt", shape="qwen3", layers=1, t=2048, start=0, prep=True),
        # a chunk of a prompt that follows cached positions
        dict(name="chunk-tinyllama-512", kind="prompt", shape="tinyllama", layers=1, t=512, start=1536, prep=False),
        # a user's next short message on a long kept conversation (prefix reuse), in
        # every layer: few rows against many keys, an odd length
        dict(name="turn-qwen2.5-12k", kind="prompt", shape="qwen2.5", layers=24, t=37, start=12001, prep=True),
        # a prompt chunk through a whole small model, logits out
        dict(name="forward-smollm2-251", kind="forward", model="smollm2-135m", t=251, start=0),
        # the greedy loop of a whole small model, then the logits where it stopped
        dict(name="greedy-smollm2-32", kind="greedy", model="smollm2-135m", start=150, steps=32),
        # a full prompt chunk through layers of a 1B model: products of 256 rows
        dict(name="forward-tinyllama-256", kind="forward", model="tinyllama-2l", t=256, start=0),
        # one token through a layer of an 8B model and its LM head: weights streamed once
        dict(name="forward-llama3-1", kind="forward", model="llama3-1l", t=1, start=700),
        # the default sampler (top-k 40, top-p 0.9) on a small vocabulary, 4 draws
        dict(name="sample-default-49k", kind="sample", vocab=49152, draws=4, temperature=0.7, top_k=40, top_p=0.9,
             min_p=0.0, penalty=1.0, history=0),
        # nucleus sampling over the whole of a large vocabulary with a repetition penalty
        dict(name="sample-nucleus-152k", kind="sample", vocab=151936, draws=4, temperature=0.8, top_k=0, top_p=0.95,
             min_p=0.0, penalty=1.1, history=600),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prompt", "prompt", "forward", "greedy", "sample"])
    if kind == "decode":
        shape = rng.choice(sorted(SHAPES))
        heads, kvh, d = SHAPES[shape][:3]
        start = _log(rng, 40, 65500)
        # up to 24 layers, the pass within the longest listed one's bytes
        layers = max(1, min(24, int(2.1e9 / (8 * start * kvh * d))))
        return dict(kind=kind, shape=shape, layers=layers, t=1, start=start, prep=rng.random() < 0.5)
    if kind == "prompt":
        shape = rng.choice(sorted(SHAPES))
        heads, kvh, d = SHAPES[shape][:3]
        t = _log(rng, 2, 2048)
        start = 0 if rng.random() < 0.4 else _log(rng, 16, 32000)
        # within the largest listed prompt's flops
        while t > 2 and 4 * d * heads * t * (start + t / 2) > 1.7e10:
            t = max(2, t * 2 // 3)
        return dict(kind=kind, shape=shape, layers=1 if t > 64 else 8, t=t, start=start, prep=rng.random() < 0.7)
    if kind == "forward":
        model = rng.choice(sorted(MODELS))
        t = 1 if rng.random() < 0.2 else _log(rng, 2, 256)
        return dict(kind=kind, model=model, t=t, start=0 if rng.random() < 0.5 else _log(rng, 16, 1500))
    if kind == "greedy":
        return dict(kind=kind, model="smollm2-135m", start=_log(rng, 8, 1500), steps=rng.randint(4, 32))
    vocab = rng.choice([32000, 49152, 128256, 151936, rng.randint(20000, 151000)])
    penalty = rng.choice([1.0, 1.1])
    return dict(kind="sample", vocab=vocab, draws=rng.randint(1, 4), temperature=rng.choice([0.6, 0.7, 0.8, 1.0]),
                top_k=rng.choice([0, 20, 40, 50, 100, 200]), top_p=rng.choice([0.9, 0.95, 1.0]),
                min_p=rng.choice([0.0, 0.0, 0.05]), penalty=penalty,
                history=_log(rng, 16, 4000) if penalty != 1.0 else 0)


# ---------------------------------------------------------------- inputs


_stream = None


def _one_stream():
    """The program's stream: what it queues runs in order, one call after another."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _inv_freq(theta, d):
    return np.array([1.0 / theta ** (2.0 * i / d) for i in range(d // 2)], np.float32)


class _Attn:
    """The inputs of an attention case, from the seed: the cached rows (RoPE already
    in them) and the new tokens' raw q, k, v, N(0, 1) as the configurations have them."""

    def __init__(self, case, seed):
        self.heads, self.kvh, self.d, self.theta, self.norm, self.bias = SHAPES[case["shape"]]
        g = _gen(seed)
        self.layers, self.t, self.start = case["layers"], case["t"], case["start"]
        self.q = torch.randn(self.layers, self.t, self.heads * self.d, generator=g, device=DEV)
        kvd = self.kvh * self.d
        self.cached = self.start if case["prep"] else self.start + self.t
        self.g, self.kvd = g, kvd
        if case["prep"]:
            self.k = torch.randn(self.layers, self.t, kvd, generator=g, device=DEV)
            self.v = torch.randn(self.layers, self.t, kvd, generator=g, device=DEV)
            n = self.heads * self.d
            self.consts = [{
                "bq": torch.randn(n, generator=g, device=DEV) * 0.3 if self.bias else None,
                "bk": torch.randn(kvd, generator=g, device=DEV) * 0.3 if self.bias else None,
                "bv": torch.randn(kvd, generator=g, device=DEV) * 0.3 if self.bias else None,
                "q_norm": 1 + 0.1 * torch.randn(self.d, generator=g, device=DEV) if self.norm else None,
                "k_norm": 1 + 0.1 * torch.randn(self.d, generator=g, device=DEV) if self.norm else None,
            } for _ in range(self.layers)]

    def cached_rows(self):
        """The next layer's cached k and v (call once per layer, in order)."""
        return (torch.randn(max(self.cached, 1), self.kvd, generator=self.g, device=DEV),
                torch.randn(max(self.cached, 1), self.kvd, generator=self.g, device=DEV))


def _config(case):
    shape, hidden, ff, layers, vocab = MODELS[case["model"]]
    heads, kvh, d, theta = SHAPES[shape][:4]
    return Config(arch="llama", hidden=hidden, intermediate=ff, layers=layers, heads=heads, kv_heads=kvh, head_dim=d,
                  vocab=vocab, max_position=8192, rms_eps=float(np.float32(1e-5)), rope_theta=theta,
                  tie_embeddings=True)


def _weights(cfg, g):
    """Random weights on the GPU: matrices N(0, 0.02), norms near 1."""
    def mat(r, c):
        return torch.randn(r, c, generator=g, device=DEV) * 0.02

    def vec(n):
        return 1 + 0.05 * torch.randn(n, generator=g, device=DEV)

    h, q, kv, ff = cfg.hidden, cfg.q_dim, cfg.kv_dim, cfg.intermediate
    w = {"embed": mat(cfg.vocab, h), "norm": vec(h), "lm_head": None, "layers": []}
    for _ in range(cfg.layers):
        w["layers"].append({"attn_norm": vec(h), "wq": mat(q, h), "wk": mat(kv, h), "wv": mat(kv, h), "wo": mat(h, q),
                            "bq": None, "bk": None, "bv": None, "q_norm": None, "k_norm": None, "ffn_norm": vec(h),
                            "w_gate": mat(ff, h), "w_up": mat(ff, h), "w_down": mat(h, ff)})
    return w


def _host(w):
    def conv(v):
        return None if v is None else v.cpu().numpy()
    return {"embed": conv(w["embed"]), "norm": conv(w["norm"]), "lm_head": None,
            "layers": [{k: conv(v) for k, v in lw.items()} for lw in w["layers"]]}


def _tokens(case, cfg, g):
    """The positions already cached and the call's own tokens."""
    n = case["start"] + (case["t"] if case["kind"] == "forward" else 0)
    ids = torch.randint(0, cfg.vocab, (n,), generator=g, device=DEV).cpu().numpy().astype(np.uint32)
    return ids[:case["start"]], ids[case["start"]:]


def _logits(case, seed):
    """Logits as a language model's are: a broad normal body and a few likely ids."""
    g = _gen(seed)
    x = torch.randn(case["draws"], case["vocab"], generator=g, device=DEV) * 2.5
    hot = torch.randint(0, case["vocab"], (case["draws"], 12), generator=g, device=DEV)
    x.scatter_add_(1, hot, torch.rand(case["draws"], 12, generator=g, device=DEV) * 4 + 4)
    hist = torch.randint(0, case["vocab"], (max(case["history"], 1),), generator=g, device=DEV).to(torch.int32)
    return x, hist


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        a = _Attn(case, seed)
        kv = DeviceKvCache(a.layers, a.start + a.t, a.kvh, a.d)
        stream = _one_stream()
        if case["prep"]:
            kv.set_rope(_inv_freq(a.theta, a.d))
            for li, c in enumerate(a.consts):
                kv.set_prep(li, a.heads, *[None if c[k] is None else c[k].cpu().numpy()
                                           for k in ("bq", "bk", "bv", "q_norm", "k_norm")], eps=1e-6)
        for li in range(a.layers):
            k, v = a.cached_rows()
            torch.cuda.synchronize()
            if a.cached:
                kv.append_device(li, 0, a.cached, k.data_ptr(), v.data_ptr())
            kv.synchronize()
        kv.set_stream(stream.cuda_stream)
        return dict(case=case, a=a, kv=kv, stream=stream, q=a.q.clone(), att=torch.empty_like(a.q))
    if kind in ("forward", "greedy"):
        cfg, g = _config(case), _gen(seed)
        w = _weights(cfg, g)
        before, toks = _tokens(case, cfg, g)
        m = DeviceModel(cfg, _host(w))
        cache = m.new_cache(case["start"] + (case["t"] if kind == "forward" else case["steps"] + 1))
        first = m.prefill(cache, before) if len(before) else None
        return dict(case=case, m=m, cache=cache, toks=toks, first=first)
    x, hist = _logits(case, seed)
    s = DeviceSampler(SamplerConfig(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"],
                                    min_p=case["min_p"], repetition_penalty=case["penalty"], seed=seed), case["vocab"])
    return dict(case=case, s=s, x=x, work=x.clone(), hist=hist,
                out=torch.zeros(case["draws"], dtype=torch.int32, device=DEV))


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        a, kv, q, att = st["a"], st["kv"], st["q"], st["att"]
        if case["prep"]:
            if a.t > 1:
                # the call prepares q in place; the products that write it each time
                # are stood for by a copy
                with torch.cuda.stream(st["stream"]):
                    q.copy_(a.q)
            for li in range(a.layers):
                kv.attend_device(li, a.heads, q[li].data_ptr(), a.k[li].data_ptr(), a.v[li].data_ptr(), a.t, a.start,
                                 att[li].data_ptr())
        else:
            for li in range(a.layers):
                kv.attention_device(li, a.heads, q[li].data_ptr(), a.t, a.start, att[li].data_ptr())
        return att
    if kind == "forward":
        st["cache"].len = case["start"]
        return st["m"].forward(st["cache"], st["toks"])
    if kind == "greedy":
        st["cache"].len = case["start"]
        ids = st["m"].decode(st["cache"], st["first"], case["steps"])
        return {"ids": np.array(ids, np.int64), "logits": st["m"].forward(st["cache"], [ids[-1]])}
    x, vocab, out = st["work"], case["vocab"], st["out"]
    if case["penalty"] != 1.0:
        x.copy_(st["x"])  # the draw penalises the logits in place; the LM head writes them anew each step
    for i in range(case["draws"]):
        st["s"].sample_device(x[i].data_ptr(), st["hist"].data_ptr(), case["history"], out[i].data_ptr())
    return {"ids": out, "logits": x}


# ---------------------------------------------------------------- what a pass cannot do without


def _pairs(t, start):
    return t * start + t * (t + 1) // 2


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        heads, kvh, d = SHAPES[case["shape"]][:3]
        t, n = case["t"], case["start"] + case["t"]
        rows = 2 * n * kvh * d + 2 * t * heads * d + (2 * t * kvh * d if case["prep"] else 0)
        return {"bytes": 4 * rows * case["layers"], "flops": 4 * d * heads * _pairs(t, case["start"]) * case["layers"]}
    if kind in ("forward", "greedy"):
        cfg = _config(case)
        q, kv, h, ff = cfg.q_dim, cfg.kv_dim, cfg.hidden, cfg.intermediate
        layer = h * (q + 2 * kv) + q * h + 3 * h * ff
        head = cfg.vocab * h
        passes = [(case["t"], case["start"])] if kind == "forward" else [
            (1, case["start"] + i) for i in range(case["steps"] + 1)]
        b = f = 0
        for t, start in passes:
            b += 4 * (cfg.layers * (layer + 2 * (start + t) * kv) + head + cfg.vocab)
            f += 2 * t * cfg.layers * layer + 2 * head + 4 * q * cfg.layers * _pairs(t, start)
        return {"bytes": b, "flops": f}
    return {"bytes": 4 * case["vocab"] * case["draws"] * (2 if case["penalty"] != 1.0 else 1),
            "flops": 4 * case["vocab"] * case["draws"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"  # wick's f32 operations in wick's order: the same ids and bits
    if kind in ("forward", "greedy"):
        return {"rel": 1e-5, "differ": 0.01}
    return {"rel": 4e-6}


# ---------------------------------------------------------------- the same in 64 bits


def _rope64(x, theta, start):
    """Rotate-half RoPE of x [t][heads][d] from position start; the angle is the f32
    product pos * inv_freq, as the reference defines it."""
    t, _, d = x.shape
    f = torch.from_numpy(_inv_freq(theta, d)).to(DEV)
    ang = (torch.arange(start, start + t, device=DEV, dtype=torch.float32)[:, None] * f[None, :]).double()
    s, c = ang.sin()[:, None, :], ang.cos()[:, None, :]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _rms64(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + float(np.float32(eps))).sqrt() * w.double()


def _attention64(q, k, v, start):
    """q [t][heads][d], k and v [n][kv_heads][d] in f64, causal from position start."""
    t, heads, d = q.shape
    n, kvh, _ = k.shape
    out = torch.empty_like(q)
    mask = torch.arange(n, device=DEV)[None, :] > start + torch.arange(t, device=DEV)[:, None]
    for h in range(heads):
        kh, vh = k[:, h // (heads // kvh)].contiguous(), v[:, h // (heads // kvh)].contiguous()
        s = q[:, h].contiguous() @ kh.t().contiguous() / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ vh
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        x, hist = _logits(case, seed)
        x = x.double()
        if case["penalty"] != 1.0 and case["history"]:
            ids, p = hist.long().unique(), float(np.float32(case["penalty"]))
            y = x[:, ids]
            x[:, ids] = torch.where(y > 0, y / p, y * p)
        return {"ids": None, "logits": x}
    if kind in ("decode", "prompt"):
        a = _Attn(case, seed)
        out = torch.empty(a.layers, a.t, a.heads * a.d, device=DEV, dtype=torch.float64)
        for li in range(a.layers):
            k, v = a.cached_rows()
            k, v = (x[:a.cached].double().reshape(-1, a.kvh, a.d) for x in (k, v))
            q = a.q[li].double().reshape(a.t, a.heads, a.d)
            if case["prep"]:
                c = a.consts[li]
                nk, nv = (x[li].double().reshape(a.t, a.kvh, a.d) for x in (a.k, a.v))
                if a.bias:
                    q = q + c["bq"].double().reshape(a.heads, a.d)
                    nk = nk + c["bk"].double().reshape(a.kvh, a.d)
                    nv = nv + c["bv"].double().reshape(a.kvh, a.d)
                if a.norm:
                    q, nk = _rms64(q, c["q_norm"], 1e-6), _rms64(nk, c["k_norm"], 1e-6)
                q, nk = _rope64(q, a.theta, a.start), _rope64(nk, a.theta, a.start)
                k, v = torch.cat([k, nk]), torch.cat([v, nv])
            out[li] = _attention64(q, k, v, a.start).reshape(a.t, -1)
        return out
    cfg, g = _config(case), _gen(seed)
    w = _weights(cfg, g)
    before, toks = _tokens(case, cfg, g)
    kc, vc = [None] * cfg.layers, [None] * cfg.layers

    def forward(ids, start):
        ids = torch.from_numpy(np.asarray(ids, np.int64)).to(DEV)
        x = w["embed"][ids].double()
        t = len(ids)
        for li, lw in enumerate(w["layers"]):
            h = _rms64(x, lw["attn_norm"], cfg.rms_eps)
            q, k, v = (h @ lw[n].double().t().contiguous() for n in ("wq", "wk", "wv"))
            q = _rope64(q.reshape(t, cfg.heads, cfg.head_dim), cfg.rope_theta, start)
            k = _rope64(k.reshape(t, cfg.kv_heads, cfg.head_dim), cfg.rope_theta, start)
            v = v.reshape(t, cfg.kv_heads, cfg.head_dim)
            kc[li] = k if start == 0 else torch.cat([kc[li], k])
            vc[li] = v if start == 0 else torch.cat([vc[li], v])
            x = x + _attention64(q, kc[li], vc[li], start).reshape(t, -1) @ lw["wo"].double().t().contiguous()
            h = _rms64(x, lw["ffn_norm"], cfg.rms_eps)
            u = torch.nn.functional.silu(h @ lw["w_gate"].double().t().contiguous())
            x = x + (u * (h @ lw["w_up"].double().t().contiguous())) @ lw["w_down"].double().t().contiguous()
        x = _rms64(x[-1:], w["norm"], cfg.rms_eps)
        return x @ w["embed"].double().t().contiguous()

    logits = forward(before, 0) if len(before) else None
    if kind == "forward":
        return forward(toks, case["start"]).cpu().numpy()
    for i in range(case["steps"] + 1):
        logits = forward([int(logits.argmax())], case["start"] + i)
    return {"ids": None, "logits": logits.cpu().numpy()}
