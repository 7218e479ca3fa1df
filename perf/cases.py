"""The measured cases: what a program that serves adapter-augmented models has this library do.

Four kinds of work, each through the public binding (aoship.py over the C ABI):

  route   a router's decisions from features (Router.route_features)
  mlp     one layer's SwiGLU MLP with its adapters: at decode routed in the same call
          (Layer.route_mlp_forward), for prompts with the rings given (Layer.mlp_forward)
  proj    one layer's attention projections: q, k and v of one input, and o (Layer.qkv_forward,
          Layer.proj_forward)
  model   token ids to logits over the KV cache (Model.forward): a prompt, or a prompt and the
          tokens decoded after it

Base weights are MLX 4-bit groups of 64 (uniform nibbles, float16 scale and bias that centre
them), LoRA weights are bfloat16 values given as float32, activations are N(0, 1) bfloat16 as
after a norm. Everything is drawn on the GPU from the seed.
"""
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "adapter-os_amd"))
import aoship  # noqa: E402

DEV = "cuda:0"
GROUP = 64
Q15 = 32767.0
EPS = 0.02  # the router's entropy floor
ROPE_THETA, RMS_EPS = 10000.0, 1e-6

MLP_7B = dict(hidden=3584, inter=18944)
ATTN_3B = dict(hidden=3072, q_out=3072, kv_out=1024)
ATTN_7B = dict(hidden=3584, q_out=3584, kv_out=512)
MODEL_7B = dict(layers=2, hidden=3584, inter=18944, heads=28, kv_heads=4, head_dim=128, vocab=32000)


def listed():
    return [
        # the decision for one decoded token: a single small launch, all latency
        dict(name="route one token", kind="route", features=3584, adapters=16, k=4, tokens=1),
        # the decisions for a whole prompt over a large adapter table, ahead of its prefill
        dict(name="route a prompt", kind="route", features=5120, adapters=64, k=8, tokens=2039),
        # one user's next token, the most frequent call of all: 7B-shaped MLP, routed in the call
        dict(name="mlp decode 1", kind="mlp", **MLP_7B, adapters=16, rank=16, k=4, tokens=1, sets=0),
        # a small batch of concurrent users
        dict(name="mlp decode 8", kind="mlp", **MLP_7B, adapters=16, rank=16, k=4, tokens=8, sets=0),
        # a busy server's decode batch, not a power of two
        dict(name="mlp decode 27", kind="mlp", **MLP_7B, adapters=16, rank=16, k=4, tokens=27, sets=0),
        # a short chat turn's prompt
        dict(name="mlp prompt 75", kind="mlp", **MLP_7B, adapters=16, rank=16, k=4, tokens=75, sets=6),
        # a long prompt whose tokens cluster on a few adapter sets
        dict(name="mlp prompt 2048", kind="mlp", **MLP_7B, adapters=16, rank=16, k=4, tokens=2048, sets=6),
        # the largest layer and adapter table: 32B-shaped, 64 adapters of rank 64, a quarter of the
        # tokens on sets of their own
        dict(name="mlp prompt 4096 wide", kind="mlp", hidden=5120, inter=27648, adapters=64, rank=64, k=8,
             tokens=4096, sets=24),
        # 32 decode streams, each with its own adapters, through a 3B-shaped layer's projections
        dict(name="proj decode 32", kind="proj", **ATTN_3B, adapters=32, rank=16, k=4, tokens=32, sets=0),
        # a ragged prompt through a 7B-shaped layer's projections
        dict(name="proj prompt 1531", kind="proj", **ATTN_7B, adapters=16, rank=16, k=4, tokens=1531, sets=6),
        # a prompt's prefill, ids to logits, through 7B-shaped decoder layers
        dict(name="model prompt 1900", kind="model", **MODEL_7B, adapters=16, rank=16, k=4, prompt=1900, steps=0),
        # a short completion: a prompt, then token by token over the cache
        dict(name="model generate", kind="model", **MODEL_7B, adapters=16, rank=16, k=4, prompt=211, steps=24),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], even over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["route", "mlp", "mlp", "mlp", "proj", "proj", "model"])
    adapters = _between(rng, 2, 64)
    k = rng.randint(1, min(8, adapters))
    if kind == "route":
        return dict(kind=kind, features=4 * _between(rng, 224, 1280), adapters=adapters, k=k,
                    tokens=_between(rng, 1, 4096))
    hidden = 64 * _between(rng, 14, 64)
    rank = rng.choice([4, 8, 12, 16, 16, 24, 32, 64])
    if kind == "model":
        hd = rng.choice([64, 64, 128, 128, 96])
        kv = rng.choice([2, 4, 8] if hd == 96 else [1, 2, 4, 8])
        heads = kv * rng.choice([1, 2, 4, 7])
        return dict(kind=kind, layers=rng.randint(1, 2), hidden=hidden, inter=64 * _between(rng, 40, 200),
                    heads=heads, kv_heads=kv, head_dim=hd, vocab=32 * _between(rng, 60, 1000),
                    adapters=min(adapters, 24), rank=min(rank, 32), k=min(k, adapters, 24), prompt=_between(rng, 1, 2048), steps=rng.choice([0, 0, rng.randint(1, 20)]))
    tokens = _between(rng, 1, 32) if rng.random() < 0.5 else _between(rng, 33, 3000)
    sets = 0 if tokens <= 32 else rng.choice([1, 4, 6, 12, 24])
    if kind == "proj":
        kv_out = 64 * _between(rng, 4, 20)
        return dict(kind=kind, hidden=hidden, q_out=kv_out * rng.choice([1, 2, 3, 7]), kv_out=kv_out,
                    adapters=adapters, rank=rank, k=k, tokens=tokens, sets=sets)
    return dict(kind=kind, hidden=hidden, inter=64 * _between(rng, 60, 320), adapters=adapters, rank=rank, k=k,
                tokens=tokens, sets=sets)


# ---- inputs from the seed -------------------------------------------------------------------------


def _gen(seed, *at):
    g = torch.Generator(device=DEV)
    v = seed
    for a in at:
        v = (v * 1000003 + a + 1) % (1 << 62)
    g.manual_seed(v)
    return g


MODULE = {m: i for i, m in enumerate(aoship.MODULES)}


def _shapes(c):
    """(out, in) of each projection of a layer."""
    h = c["hidden"]
    s = {}
    if c["kind"] != "mlp":
        qo = c["q_out"] if c["kind"] == "proj" else c["heads"] * c["head_dim"]
        kvo = c["kv_out"] if c["kind"] == "proj" else c["kv_heads"] * c["head_dim"]
        s.update(q_proj=(qo, h), k_proj=(kvo, h), v_proj=(kvo, h), o_proj=(h, qo))
    if c["kind"] != "proj":
        s.update(gate_proj=(c["inter"], h), up_proj=(c["inter"], h), down_proj=(h, c["inter"]))
    return s


def _q4(seed, at, out, inp):
    """A 4-bit matrix: packed [out, in/8] int32, scale and bias [out, in/64] float16 (on the GPU)."""
    g = _gen(seed, 1, *at)
    packed = torch.randint(-(1 << 31), 1 << 31, (out, inp // 8), generator=g, device=DEV, dtype=torch.int32)
    n = (out, inp // GROUP)
    scale = (0.0040 * (0.75 + 0.5 * torch.rand(n, generator=g, device=DEV))).half()
    bias = (-scale.float() * (7.5 + 0.2 * torch.randn(n, generator=g, device=DEV))).half()
    return packed, scale, bias


def _host(packed, scale, bias):
    return packed.cpu().numpy().view(np.uint32), scale.cpu().numpy(), bias.cpu().numpy()


def _lora(seed, layer, module, n, rank, out, inp):
    """All adapters' A [n, rank, in] and B [n, out, rank]: bfloat16 values as float32 (on the GPU)."""
    g = _gen(seed, 2, layer, MODULE[module])
    a = torch.randn((n, rank, inp), generator=g, device=DEV) * inp ** -0.5
    b = torch.randn((n, out, rank), generator=g, device=DEV) * 0.02
    return a.bfloat16().float(), b.bfloat16().float()


def _x(seed, at, *shape):
    return torch.randn(shape, generator=_gen(seed, 3, at), device=DEV).bfloat16()


def _features(c, seed):
    d = c.get("features", c.get("hidden"))
    f = torch.randn((c["tokens"], d), generator=_gen(seed, 4), device=DEV)
    w = torch.randn((c["adapters"], d), generator=_gen(seed, 5), device=DEV) * 0.05
    return f, w


def _rings(c, seed, tokens, sets):
    """The decisions a router hands over for a prompt: most tokens on one of `sets` adapter sets, one
    in four (with few sets: none) on a set of its own; with sets = 0 every token on its own. Returns
    the adapters [tokens, k] and the Q15 gates [tokens, k], largest first, on the GPU."""
    n, k = c["adapters"], c["k"]
    g = _gen(seed, 6)
    own = torch.rand((tokens, n), generator=g, device=DEV)
    score = own
    if sets:
        shared = torch.rand((sets, n), generator=g, device=DEV)
        pick = torch.randint(0, sets, (tokens,), generator=g, device=DEV)
        alone = torch.rand((tokens,), generator=g, device=DEV) < (0.25 if sets > 12 else 0.0)
        score = torch.where(alone[:, None], own, shared[pick])
    ids = torch.argsort(score, dim=1, descending=True, stable=True)[:, :k]
    logits = torch.randn((tokens, k), generator=g, device=DEV).double().sort(dim=1, descending=True).values
    return ids, _gates(logits, k)


def _gates(logits, k):
    p = torch.softmax(logits, dim=1).clamp_min(EPS / k)
    return torch.floor(p / p.sum(dim=1, keepdim=True) * Q15 + 0.5)


def _ring_bytes(ids, gates):
    """aoship_ring_t of every token, as device bytes."""
    t, k = ids.shape
    r = np.zeros(t, aoship.RING_DTYPE)
    r["top_k"] = k
    r["current_pos"] = 0
    r["adapter_indices"][:, :k] = ids.cpu().numpy()
    r["gates_q15"][:, :k] = gates.cpu().numpy()
    return torch.from_numpy(r.view(np.uint8).copy()).to(DEV)


def _set_lora(adapters, c, seed, layer):
    for m, (out, inp) in _shapes(c).items():
        a, b = (t.cpu().numpy() for t in _lora(seed, layer, m, len(adapters), c["rank"], out, inp))
        for i, ad in enumerate(adapters):
            ad.set_module(layer, m, a[i], b[i])


def _norm_weight(seed, at, h):
    return 1.0 + 0.1 * torch.randn(h, generator=_gen(seed, 7, at), device=DEV)


def _model_inputs(c, seed):
    t = c["prompt"] + c["steps"]
    ids = torch.randint(0, c["vocab"], (t,), generator=_gen(seed, 8), device=DEV, dtype=torch.int32)
    return ids, _rings(c, seed, t, 6)


def prepare(case, seed):
    c = case
    aoship.init(0)
    if c["kind"] == "route":
        f, w = _features(c, seed)
        ids = np.arange(c["adapters"], dtype=np.uint64)
        return dict(case=c, f=f, w=w, router=aoship.Router(c["adapters"], c["k"], 1.0, EPS, 1.0, ids),
                    rings=torch.zeros(c["tokens"] * 40, dtype=torch.uint8, device=DEV),
                    priors=torch.zeros((c["tokens"], c["adapters"]), device=DEV),
                    status=torch.zeros(c["tokens"], dtype=torch.int32, device=DEV))
    layers = c.get("layers", 1)
    adapters = [aoship.LoraAdapter(i, layers, 1.0) for i in range(c["adapters"])]
    for i in range(layers):
        _set_lora(adapters, c, seed, i)
    if c["kind"] == "model":
        m = aoship.Model(layers, c["hidden"], c["inter"], c["heads"], c["kv_heads"], c["head_dim"], c["vocab"],
                         c["prompt"] + c["steps"], ROPE_THETA, RMS_EPS)
        for i, layer in enumerate(m.layers):
            for name, (out, inp) in _shapes(c).items():
                layer.set_base(name, *_host(*_q4(seed, (i, MODULE[name]), out, inp)))
            for which in (0, 1):
                m.set_norm(i, which, _norm_weight(seed, 2 * i + which, c["hidden"]).cpu().numpy())
        m.set_norm(-1, 0, _norm_weight(seed, 99, c["hidden"]).cpu().numpy())
        m.set_embedding(*_host(*_embedding(c, seed)))
        m.set_lm_head(*_host(*_q4(seed, (98, 1), c["vocab"], c["hidden"])))
        m.set_adapters(adapters)
        m.reserve(max(1, c["prompt"]))
        ids, rings = _model_inputs(c, seed)
        return dict(case=c, model=m, ids=ids, rings=_ring_bytes(*rings),
                    logits=torch.zeros((1 + c["steps"], c["vocab"]), device=DEV))
    layer = aoship.Layer(0)
    for name, (out, inp) in _shapes(c).items():
        layer.set_base(name, *_host(*_q4(seed, (0, MODULE[name]), out, inp)))
    layer.set_adapters(adapters)
    layer.reserve(c["tokens"])
    t, h = c["tokens"], c["hidden"]
    s = dict(case=c, layer=layer, x=_x(seed, 0, t, h), y=torch.empty((t, h), dtype=torch.bfloat16, device=DEV))
    if c["kind"] == "proj":
        s["rings"] = _ring_bytes(*_rings(c, seed, t, c["sets"]))
        s["attn"] = _x(seed, 1, t, c["q_out"])
        for n, w in (("q", c["q_out"]), ("k", c["kv_out"]), ("v", c["kv_out"])):
            s[n] = torch.empty((t, w), dtype=torch.bfloat16, device=DEV)
    elif c["sets"] == 0:  # decode: routed in the call
        s["f"], s["w"] = _features(c, seed)
        s["router"] = aoship.Router(c["adapters"], c["k"], 1.0, EPS, 1.0, np.arange(c["adapters"], dtype=np.uint64))
        s["rings"] = torch.zeros(t * 40, dtype=torch.uint8, device=DEV)
    else:
        s["rings"] = _ring_bytes(*_rings(c, seed, t, c["sets"]))
    return s


def _embedding(c, seed):
    """Embedding rows of about unit size."""
    packed, scale, bias = _q4(seed, (98, 0), c["vocab"], c["hidden"])
    return packed, scale * 48, bias * 48


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "route":
        s["router"].route_features(s["f"], s["w"], s["rings"], s["priors"], s["status"])
        return dict(rings=s["rings"], priors=s["priors"], status=s["status"])
    if c["kind"] == "proj":
        s["layer"].qkv_forward(s["x"], s["rings"], s["q"], s["k"], s["v"])
        s["layer"].proj_forward("o_proj", s["attn"], s["rings"], s["y"])
        return dict(q=s["q"], k=s["k"], v=s["v"], o=s["y"])
    if c["kind"] == "model":
        m, p = s["model"], c["prompt"]
        m.reset_cache()
        m.forward(s["ids"][:p], s["rings"][: 40 * p], s["logits"][0])
        for i in range(c["steps"]):
            m.forward(s["ids"][p + i : p + i + 1], s["rings"][40 * (p + i) : 40 * (p + i + 1)], s["logits"][1 + i])
        return s["logits"]
    if c["sets"] == 0:
        s["layer"].route_mlp_forward(s["router"], s["f"], s["w"], s["x"], s["rings"], s["y"])
        return dict(y=s["y"], rings=s["rings"])
    s["layer"].mlp_forward(s["x"], s["rings"], s["y"])
    return s["y"]


# ---- the least work of a pass -----------------------------------------------------------------------


def _layer_work(c, tokens):
    """Bytes and operations of one layer's projections for `tokens` tokens: the base weights, the rows of
    the adapters that the tokens can use, the operations of the base product and the K deltas."""
    used = min(c["adapters"], c["k"] * max(1, tokens if not c.get("sets", 6) or c.get("sets", 6) > 12 else c.get("sets", 6)))
    nbytes = flops = 0
    for out, inp in _shapes(c).values():
        nbytes += out * inp // 2 + 4 * out * (inp // GROUP) + 2 * used * c["rank"] * (out + inp)
        flops += 2 * tokens * (out * inp + c["k"] * c["rank"] * (out + inp))
    return nbytes, flops


def work(case):
    c = case
    if c["kind"] == "route":
        t, n, d = c["tokens"], c["adapters"], c["features"]
        return {"bytes": 4 * (t * d + n * d + t * n) + 44 * t, "flops": 2 * t * n * d}
    if c["kind"] == "model":
        nbytes = flops = 0
        kv = 2 * c["layers"] * c["kv_heads"] * c["head_dim"] * 2  # cache bytes of a position
        qd = c["heads"] * c["head_dim"]
        p = c["prompt"]
        for t, seen in [(p, p)] + [(1, p + 1 + i) for i in range(c["steps"])]:
            b, f = _layer_work(c, t)
            pairs = t * (seen - t) + t * (t + 1) // 2
            nbytes += c["layers"] * b + kv * seen + t * c["hidden"] // 2
            flops += c["layers"] * (f + 4 * pairs * qd)
            nbytes += c["vocab"] * c["hidden"] // 2 + 4 * c["vocab"] * (c["hidden"] // GROUP) + 4 * c["vocab"]
            flops += 2 * c["vocab"] * c["hidden"]
        return {"bytes": nbytes, "flops": flops}
    t, h = c["tokens"], c["hidden"]
    nbytes, flops = _layer_work(c, t)
    if c["kind"] == "proj":
        nbytes += 2 * t * (2 * h + 2 * c["q_out"] + 2 * c["kv_out"]) + 40 * t
    else:
        nbytes += 4 * t * h + 40 * t
        if c["sets"] == 0:
            nbytes += 4 * h * (t + c["adapters"])
            flops += 2 * t * c["adapters"] * h
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    c = case
    if c["kind"] == "route":
        return "exact"  # decisions are deterministic, and the priors' order of summation is part of the interface
    if c["kind"] == "proj":
        return {"rel": 4e-3, "max": 0.03}  # one bfloat16 rounding of the result
    if c["kind"] == "mlp":
        return {"rel": 8e-3, "max": 0.1}  # the rounding of h (bfloat16), then of the result
    return {"rel": 0.02, "max": 0.3}  # the roundings of up to two decoder layers


# ---- the same in 64 bits ----------------------------------------------------------------------------


def _dense(packed, scale, bias):
    out, w = packed.shape
    q = (packed[:, :, None] >> (4 * torch.arange(8, device=DEV, dtype=torch.int32))) & 15
    q = q.reshape(out, -1, GROUP).double()
    return (q * scale.double()[:, :, None] + bias.double()[:, :, None]).reshape(out, 8 * w)


def _linear(c, seed, layer, module, x, ids, gates):
    out, inp = _shapes(c)[module]
    y = x @ _dense(*_q4(seed, (layer, MODULE[module]), out, inp)).T
    a, b = _lora(seed, layer, module, c["adapters"], c["rank"], out, inp)
    for i in range(c["adapters"]):
        coef = ((ids == i) * gates.double()).sum(dim=1) / Q15
        at = coef.nonzero()[:, 0]
        if at.numel():
            y[at] += coef[at, None] * ((x[at] @ a[i].double().T) @ b[i].double().T)
    return y


def _mlp(c, seed, layer, x, ids, gates):
    g = _linear(c, seed, layer, "gate_proj", x, ids, gates)
    h = g * torch.sigmoid(g) * _linear(c, seed, layer, "up_proj", x, ids, gates)
    return _linear(c, seed, layer, "down_proj", h, ids, gates)


def _route(c, f, w):
    priors = f.double() @ w.double().T
    top = torch.sort(priors, dim=1, descending=True, stable=True)
    return priors, top.indices[:, : c["k"]], _gates(top.values[:, : c["k"]], c["k"])


def _rope(x):
    """Halves rotated by position times frequency; the angle is a float32 product and the frequencies are
    float32, as the model defines them."""
    t, _, hd = x.shape
    e = np.float32(-2.0) * np.arange(hd // 2, dtype=np.float32) / np.float32(hd)
    inv = np.float32(1.0) / np.power(np.float64(ROPE_THETA), e.astype(np.float64)).astype(np.float32)
    ang = np.arange(t, dtype=np.float32)[:, None] * inv[None, :]
    ang = torch.from_numpy(ang.astype(np.float64)).to(DEV)[:, None, :]
    x1, x2 = x[..., : hd // 2], x[..., hd // 2 :]
    return torch.cat([x1 * ang.cos() - x2 * ang.sin(), x1 * ang.sin() + x2 * ang.cos()], dim=-1)


def _rms(x, w):
    return x * (w.double() / torch.sqrt((x * x).mean(dim=1, keepdim=True) + RMS_EPS))


def _model(c, seed):
    ids, (ring_ids, gates) = _model_inputs(c, seed)
    t, nh, nkv, hd = ids.numel(), c["heads"], c["kv_heads"], c["head_dim"]
    e = _embedding(c, seed)
    hid = _dense(*(v[ids.long()] for v in e))
    later = torch.triu(torch.ones((t, t), dtype=torch.bool, device=DEV), 1)
    for i in range(c["layers"]):
        x = _rms(hid, _norm_weight(seed, 2 * i, c["hidden"]))
        q, k, v = (_linear(c, seed, i, m, x, ring_ids, gates) for m in ("q_proj", "k_proj", "v_proj"))
        q, k, v = _rope(q.view(t, nh, hd)), _rope(k.view(t, nkv, hd)), v.view(t, nkv, hd)
        o = torch.empty((t, nh, hd), dtype=torch.float64, device=DEV)
        for h in range(nh):
            s = (q[:, h] @ k[:, h // (nh // nkv)].T) * hd ** -0.5
            o[:, h] = torch.softmax(s.masked_fill(later, -torch.inf), dim=1) @ v[:, h // (nh // nkv)]
        hid = hid + _linear(c, seed, i, "o_proj", o.view(t, nh * hd), ring_ids, gates)
        x = _rms(hid, _norm_weight(seed, 2 * i + 1, c["hidden"]))
        hid = hid + _mlp(c, seed, i, x, ring_ids, gates)
    last = hid[c["prompt"] - 1 :]
    return _rms(last, _norm_weight(seed, 99, c["hidden"])) @ _dense(*_q4(seed, (98, 1), c["vocab"], c["hidden"])).T


def exact(case, seed):
    c = case
    if c["kind"] == "route":
        return dict(rings=None, priors=_route(c, *_features(c, seed))[0], status=None)
    if c["kind"] == "model":
        return _model(c, seed)
    t, h = c["tokens"], c["hidden"]
    x = _x(seed, 0, t, h).double()
    if c["kind"] == "proj":
        ids, gates = _rings(c, seed, t, c["sets"])
        out = {n: _linear(c, seed, 0, n + "_proj", x, ids, gates) for n in "qkv"}
        out["o"] = _linear(c, seed, 0, "o_proj", _x(seed, 1, t, c["q_out"]).double(), ids, gates)
        return out
    if c["sets"] == 0:
        _, ids, gates = _route(c, *_features(c, seed))
        return dict(y=_mlp(c, seed, 0, x, ids, gates), rings=None)
    ids, gates = _rings(c, seed, t, c["sets"])
    return _mlp(c, seed, 0, x, ids, gates)
