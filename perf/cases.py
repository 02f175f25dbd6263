"""What this framework is used for, as cases that can be timed and compared.

Four kinds of case, each a call of a public entry point:

  layer      MoeLayer.feed_forward: the routed layer (router, dispatch, SwiGLU
             experts, combine, shared expert) over t tokens; "tiled" says
             whether the program keeps the tiled expert copies
             (MoeLayer.set_tiled), as the bench does, or not, as Model does.
             One expert and no choice is a dense MLP.
  linear     Linear: a plain projection (attention's q/k/v/o, the latent
             projections, lm_head) over t tokens
  attention  moe_attention: causal attention of many sequences over their
             f32 caches, one row per sequence (decode) or runs of rows
             (prefill), grouped heads, windows, wide keys
  model      Model.forward: a whole decoder step, its logits

Weights are N(0, 0.02) values in the stored block formats, activations
N(0, 1) as they leave a norm; everything is made on the GPU from the seed.
`exact` recomputes each case in 64 bits with torch alone.
"""
import ctypes
import math

import numpy as np
import torch

from moe_amd import _lib, synth
from moe_amd.layer import Context, MoeLayer, MoeSpec, Rec, Store, View
from moe_amd.model import HostCheckpoint, HostTensor, Linear, Model, Spec, upload_store

F32, Q4_0, Q5_0, Q8_0 = 0, 2, 6, 8
BLOCK_BYTES = {Q4_0: 18, Q5_0: 22, Q8_0: 34}
WEIGHT_STD = 0.02
DEV = "cuda:0"


# ------------------------------------------------------------------ the cases


def layer_case(shape, t, tiled):
    """A synth.Shape's fields as plain values."""
    s = synth.SHAPES[shape]
    return {"kind": "layer", "hidden": s.hidden, "inter": s.inter, "experts": s.n_experts, "top_k": s.top_k,
            "dt": s.expert_dt, "sigmoid": s.sigmoid, "norm_topk": s.norm_topk, "scale": s.routed_scale,
            "groups": s.n_group, "topk_groups": s.topk_group, "shared": s.shared_inter,
            "shared_dt": s.shared_dt if s.shared_dt is not None else s.expert_dt, "shared_gate": s.shared_gate,
            "bias_std": s.e_bias_std, "t": t, "tiled": tiled}


def listed():
    return [
        # One user's decode step through a layer of few large experts: the
        # latency that single-stream generation is made of.
        dict(layer_case("mixtral", 1, False), name="mixtral_t1"),
        # The same for many small experts behind a group-limited sigmoid
        # router with a shared expert in another format.
        dict(layer_case("deepseek_v3", 1, False), name="deepseek_v3_t1"),
        # Batched decode: 32 sequences, the tiled copies kept.
        dict(layer_case("mixtral", 32, True), name="mixtral_t32"),
        # Batched decode inside Model (which keeps no tiled copies): 32
        # sequences, 64 experts and a shared expert, 8-bit weights.
        dict(layer_case("v2_lite", 32, False), name="v2_lite_t32"),
        # Prefill of one prompt of ordinary length.
        dict(layer_case("mixtral", 512, True), name="mixtral_t512"),
        # Prefill over many small experts, a length off every tile.
        dict(layer_case("qwen3", 2041, False), name="qwen3_t2041"),
        # The largest call: 256 experts, a long prompt.
        dict(layer_case("deepseek_v3", 4096, False), name="deepseek_v3_t4096"),
        # The smallest call: one token through an attention projection.
        {"name": "q_proj_t1", "kind": "linear", "rows": 3072, "cols": 2048, "dt": Q8_0, "t": 1},
        # The head over a decode batch: the widest projection there is.
        {"name": "lm_head_t32", "kind": "linear", "rows": 102400, "cols": 2048, "dt": Q8_0, "t": 32},
        # A decode step's attention: 32 sequences of differing lengths, 16
        # heads with keys of 192 and values of 128 (latent attention's
        # expanded cache).
        {"name": "attn_decode", "kind": "attention", "seqs": 32, "new": 1, "past": 900, "heads": 16, "kv_heads": 16,
         "qd": 192, "vd": 128, "window": 0},
        # A prompt's attention: one sequence, 32 heads over 8 key/value heads.
        {"name": "attn_prefill", "kind": "attention", "seqs": 1, "new": 1000, "past": 0, "heads": 32, "kv_heads": 8,
         "qd": 128, "vd": 128, "window": 0},
        # A whole decode step of a small model, four sequences.
        {"name": "model_decode", "kind": "model", "seqs": 4, "new": 1, "past": 96},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "linear", "linear", "attention", "attention", "model"])
    if kind == "layer":
        name = rng.choice(["mixtral", "qwen3", "deepseek_v3", "v2_lite", "qwen2_moe", "tiny_mixtral"])
        c = layer_case(name, _log(rng, 1, 2048), rng.random() < 0.5)
        # The formats of the same models as other checkpoints hold them, and
        # experts somewhat narrower or wider.
        c["dt"] = rng.choice([Q4_0, Q5_0, Q8_0])
        c["shared_dt"] = rng.choice([c["dt"], c["shared_dt"]])
        c["inter"] = 64 * rng.randint(c["inter"] // 128, c["inter"] // 64)
        if rng.random() < 0.15:  # a dense MLP
            c.update(experts=1, top_k=1, groups=1, topk_groups=1, shared=0, shared_gate=False, bias_std=0.0,
                     sigmoid=False, norm_topk=True, scale=1.0)
        return c
    if kind == "linear":
        rows, cols = rng.choice([(3072, 2048), (576, 2048), (4096, 512), (2048, 2048), (32000, 512), (102400, 2048),
                                 (4096, 4096), (1024, 4096), (768, 512)])
        return {"kind": "linear", "rows": rows, "cols": cols, "dt": rng.choice([Q4_0, Q5_0, Q8_0, Q8_0]),
                "t": _log(rng, 1, 256 if rows > 50000 else 2048)}
    if kind == "attention":
        heads, kv, qd, vd = rng.choice([(16, 16, 192, 128), (8, 2, 64, 64), (32, 8, 128, 128), (32, 4, 128, 128),
                                        (16, 2, 80, 80), (4, 4, 40, 24)])
        c = {"kind": "attention", "heads": heads, "kv_heads": kv, "qd": qd, "vd": vd,
             "window": _log(rng, 16, 512) if rng.random() < 0.25 else 0}
        how = rng.randrange(3)
        if how == 0:    # decode
            c.update(seqs=_log(rng, 1, 48), new=1, past=_log(rng, 1, 2000))
        elif how == 1:  # prefill of one or a few prompts
            c.update(seqs=rng.randint(1, 4), new=_log(rng, 2, 1000), past=0)
        else:           # a chunk of a prompt behind a longer past
            c.update(seqs=rng.randint(1, 8), new=_log(rng, 2, 128), past=_log(rng, 1, 1500))
        return c
    new = rng.choice([1, 1, _log(rng, 2, 64)])
    return {"kind": "model", "seqs": _log(rng, 1, 32), "new": new, "past": 0 if new > 1 else _log(rng, 1, 128)}


# --------------------------------------------------------------- stored weights


def _generator(seed, salt):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _quantise(w, dt):
    """Rows of 32-value blocks as their stored bytes (w: f32 [n, 32])."""
    n = w.shape[0]
    if dt == Q8_0:
        d = (w.abs().amax(1) / 127.0).half()
        q = torch.round(w / d.float().clamp_min(1e-30)[:, None]).clamp_(-127, 127).to(torch.int8)
        return torch.cat([d.view(torch.uint8).view(n, 2), q.view(torch.uint8)], 1)
    top = 8 if dt == Q4_0 else 16
    far = w.gather(1, w.abs().argmax(1, keepdim=True))[:, 0]
    d = (far / -float(top)).half()
    inv = torch.where(d == 0, torch.zeros_like(far), 1.0 / d.float())
    q = torch.floor(w * inv[:, None] + (top + 0.5)).clamp_(0, 2 * top - 1).to(torch.uint8)
    low = q & 15
    codes = low[:, :16] | (low[:, 16:] << 4)
    head = [d.view(torch.uint8).view(n, 2)]
    if dt == Q5_0:
        bits = (q >> 4).view(n, 4, 8)
        weight = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=w.device)
        head.append((bits * weight).sum(2, dtype=torch.uint8))
    return torch.cat(head + [codes], 1)


def _stored(seed, salt, dt, rows, cols):
    """The stored bytes of a [rows, cols] matrix of N(0, 0.02) values."""
    blocks = rows * cols // 32
    out = torch.empty((blocks, BLOCK_BYTES[dt]), dtype=torch.uint8, device=DEV)
    g = _generator(seed, salt)
    step = 1 << 22
    for a in range(0, blocks, step):
        n = min(step, blocks - a)
        out[a:a + n] = _quantise(torch.randn((n, 32), generator=g, device=DEV) * WEIGHT_STD, dt)
    return out.view(-1)


def _values(raw, dt, rows, cols):
    """The 64-bit values of stored bytes (quantisation's definition)."""
    b = raw.view(rows * cols // 32, BLOCK_BYTES[dt])
    d = b[:, :2].contiguous().view(torch.float16).double()
    if dt == Q8_0:
        q = b[:, 2:].contiguous().view(torch.int8).double()
    else:
        codes = b[:, -16:]
        q = torch.cat([codes & 15, codes >> 4], 1)
        if dt == Q5_0:
            at = torch.arange(8, device=b.device, dtype=torch.uint8)
            q = q | (((b[:, 2:6, None] >> at) & 1) << 4).view(-1, 32)
        q = q.double() - (8 if dt == Q4_0 else 16)
    return (q * d).view(rows, cols)


def _normal(seed, salt, shape, std=1.0):
    return torch.randn(shape, generator=_generator(seed, salt), device=DEV) * std


class _Bytes:
    """Device memory of an uploaded region, for torch to fill."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "|u1", "data": (ptr, False), "version": 3}


def _region(ctx, parts):
    """Parts (uint8 tensors) in one region, each on a 256-byte boundary."""
    offs, end = [], 0
    for p in parts:
        offs.append(end)
        end = (end + p.numel() + 255) // 256 * 256
    region = ctx.upload(np.zeros(end, dtype=np.uint8))
    mem = torch.as_tensor(_Bytes(region.device_ptr(), end), device=DEV)
    for p, o in zip(parts, offs):
        mem[o:o + p.numel()] = p
    return region, offs


# ------------------------------------------------------------------------ layer


def _layer_bytes(c, seed):
    """Stored tensors of a layer by name: (format, slabs, rows, cols, bytes)."""
    E, H, I, S = c["experts"], c["hidden"], c["inter"], c["shared"]
    raw = lambda x: x.contiguous().view(torch.uint8).view(-1)  # noqa: E731
    router = torch.zeros((1, H), device=DEV) if E == 1 else _normal(seed, 1, (E, H), WEIGHT_STD)
    out = {"router": (F32, 1, E, H, raw(router))}
    if c["bias_std"] > 0:
        out["e_bias"] = (F32, 1, 1, E, raw(_normal(seed, 2, (E,), c["bias_std"])))
    for i, (name, r, k) in enumerate((("gate", I, H), ("up", I, H), ("down", H, I))):
        out["experts." + name] = (c["dt"], E, r, k, _stored(seed, 10 + i, c["dt"], E * r, k))
    if S:
        for i, (name, r, k) in enumerate((("gate", S, H), ("up", S, H), ("down", H, S))):
            out["shared." + name] = (c["shared_dt"], 1, r, k, _stored(seed, 20 + i, c["shared_dt"], r, k))
    if c["shared_gate"]:
        out["shared_gate"] = (F32, 1, 1, H, raw(_normal(seed, 3, (H,), WEIGHT_STD)))
    return out


def _prepare_layer(c, seed):
    ctx = Context(0)
    E, H, I = c["experts"], c["hidden"], c["inter"]
    tensors = _layer_bytes(c, seed)
    region, offs = _region(ctx, [v[4] for v in tensors.values()])
    store = Store(region, {n: Rec(*v[:4], o) for (n, v), o in zip(tensors.items(), offs)})
    experts = [(store.view("experts.gate", e, 0, I), store.view("experts.up", e, 0, I),
                store.view("experts.down", e, 0, H)) for e in range(E)]
    spec = MoeSpec(hidden=H, n_experts=E, top_k=c["top_k"], sigmoid=c["sigmoid"], norm_topk=c["norm_topk"],
                   routed_scale=c["scale"], n_group=c["groups"], topk_group=c["topk_groups"])
    shared = tuple(store.get("shared." + n) for n in ("gate", "up", "down")) if c["shared"] else None
    torch.cuda.synchronize()  # the region's bytes are there before the layer reads their scales
    layer = MoeLayer(ctx, spec, store.get("router"), experts, e_bias=store.get("e_bias"), shared=shared,
                     shared_gate=store.get("shared_gate"))
    if c["tiled"]:
        layer.set_tiled(True)
    x = _normal(seed, 30, (c["t"], H))
    return {"layer": layer, "ctx": ctx, "x": x, "out": torch.empty_like(x)}


def _run_layer(s):
    s["layer"].feed_forward(s["x"], s["out"])
    return s["out"]


def _route(c, t, x):
    """Expert ids and weights [T, k] (64-bit) from the stored router."""
    E = c["experts"]
    router = t["router"][4].view(torch.float32).view(E, -1).double()
    logits = x @ router.T
    score = torch.sigmoid(logits) if c["sigmoid"] else torch.softmax(logits, 1)
    rank = score + (t["e_bias"][4].view(torch.float32).double() if "e_bias" in t else 0.0)
    if c["groups"] > 1 and c["topk_groups"] < c["groups"]:
        by = rank.view(len(x), c["groups"], -1)
        best = by.topk(min(2, by.shape[2]), 2).values.sum(2).topk(c["topk_groups"], 1).indices
        keep = torch.zeros((len(x), c["groups"]), dtype=torch.bool, device=x.device).scatter_(1, best, True)
        rank = by.masked_fill(~keep[:, :, None], -math.inf).view(len(x), E)
    sel = rank.topk(min(c["top_k"], E), 1).indices
    w = score.gather(1, sel)
    if c["norm_topk"]:
        w = w / w.sum(1, keepdim=True).clamp_min(1e-20)
    return sel, w * c["scale"]


def _swiglu(x, gate, up, down):
    return (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T


def _slab(tensor, e):
    dt, slabs, rows, cols, raw = tensor
    n = raw.numel() // slabs
    return _values(raw[e * n:(e + 1) * n], dt, rows, cols)


def _exact_layer(c, seed):
    t = _layer_bytes(c, seed)
    x = _normal(seed, 30, (c["t"], c["hidden"])).double()
    sel, w = _route(c, t, x)
    out = torch.zeros_like(x)
    for e in torch.unique(sel).tolist():
        tok, slot = (sel == e).nonzero(as_tuple=True)
        y = _swiglu(x[tok], *(_slab(t["experts." + n], e) for n in ("gate", "up", "down")))
        out.index_add_(0, tok, y * w[tok, slot][:, None])
    if c["shared"]:
        y = _swiglu(x, *(_slab(t["shared." + n], 0) for n in ("gate", "up", "down")))
        if c["shared_gate"]:
            y = y * torch.sigmoid(x @ t["shared_gate"][4].view(torch.float32).double())[:, None]
        out += y
    return out


def _stored_bytes(dt, values):
    return values // 32 * BLOCK_BYTES[dt]


def _work_layer(c):
    t, E, H, I, S = c["t"], c["experts"], c["hidden"], c["inter"], c["shared"]
    k = min(c["top_k"], E)
    # Experts that t tokens of k distinct experts each are expected to reach.
    hit = E * (1.0 - (1.0 - k / E) ** t)
    weights = hit * _stored_bytes(c["dt"], 3 * H * I) + _stored_bytes(c["shared_dt"], 3 * H * S) + 4 * E * H
    return {"bytes": int(weights + 8 * t * H), "flops": 2 * t * (E * H + 3 * H * (k * I + S))}


# ----------------------------------------------------------------------- linear


def _prepare_linear(c, seed):
    ctx = Context(0)
    region, offs = _region(ctx, [_stored(seed, 40, c["dt"], c["rows"], c["cols"])])
    torch.cuda.synchronize()
    lin = Linear(ctx, View(c["dt"], c["rows"], c["cols"], region.id, offs[0]))
    ws = MoeLayer.new_workspace(lin.workspace_size(c["t"]))
    return {"lin": lin, "ctx": ctx, "ws": ws, "x": _normal(seed, 41, (c["t"], c["cols"])),
            "y": torch.empty((c["t"], c["rows"]), device=DEV)}


def _run_linear(s):
    return s["lin"](s["x"], s["y"], s["ws"])


def _exact_linear(c, seed):
    w = _values(_stored(seed, 40, c["dt"], c["rows"], c["cols"]), c["dt"], c["rows"], c["cols"])
    return _normal(seed, 41, (c["t"], c["cols"])).double() @ w.T


def _work_linear(c):
    n, k, t = c["rows"], c["cols"], c["t"]
    return {"bytes": _stored_bytes(c["dt"], n * k) + 4 * t * (n + k), "flops": 2 * t * n * k}


# -------------------------------------------------------------------- attention


def _past(c, s):
    """Cached positions of sequence s before the call: lengths differ from
    sequence to sequence, between half and one and a half times c["past"]."""
    return c["past"] * (16 + (7 * s) % 17) // 24 if c["seqs"] > 1 else c["past"]


def _attention_inputs(c, seed):
    ctx = max(_past(c, s) for s in range(c["seqs"])) + c["new"]
    q = _normal(seed, 50, (c["seqs"] * c["new"], c["heads"] * c["qd"]))
    kc = _normal(seed, 51, (c["seqs"], ctx, c["kv_heads"] * c["qd"]))
    vc = _normal(seed, 52, (c["seqs"], ctx, c["kv_heads"] * c["vd"]))
    seq = [s for s in range(c["seqs"]) for _ in range(c["new"])]
    pos = [_past(c, s) + i for s in range(c["seqs"]) for i in range(c["new"])]
    return q, kc, vc, seq, pos


def _prepare_attention(c, seed):
    q, kc, vc, seq, pos = _attention_inputs(c, seed)
    put = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    return {"c": dict(c), "q": q, "kc": kc, "vc": vc, "seq": put(seq), "pos": put(pos), "max_pos": max(pos),
            "out": torch.empty((len(seq), c["heads"] * c["vd"]), device=DEV)}


def _run_attention(s):
    c, q, out, p = s["c"], s["q"], s["out"], ctypes.c_void_p
    rc = _lib.lib().moe_attention(p(q.data_ptr()), q.shape[1], q.shape[0], c["heads"], c["kv_heads"], c["qd"], c["vd"],
                                  1.0 / math.sqrt(c["qd"]), p(s["kc"].data_ptr()), p(s["vc"].data_ptr()),
                                  s["kc"].shape[1], p(s["seq"].data_ptr()), p(s["pos"].data_ptr()), s["max_pos"],
                                  c["window"], p(out.data_ptr()), out.shape[1],
                                  p(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "moe_attention")
    return out


def _attend(q, k, v, first, window):
    """q [n, heads, qd] at positions first.. over k, v [m, kv, d], 64-bit."""
    n, heads, qd = q.shape
    rep = heads // k.shape[1]
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = torch.stack([q[:, h] @ k[:, h].T for h in range(heads)]) * np.float64(np.float32(1.0 / math.sqrt(qd)))
    at = first + torch.arange(n, device=q.device)[:, None] - torch.arange(k.shape[0], device=q.device)[None, :]
    hide = (at < 0) | ((at >= window) if window > 0 else torch.zeros_like(at, dtype=torch.bool))
    w = torch.softmax(s.masked_fill(hide, -math.inf), 2)
    return torch.stack([w[h] @ v[:, h] for h in range(heads)], 1)


def _exact_attention(c, seed):
    q, kc, vc, _, _ = _attention_inputs(c, seed)
    q = q.double().view(c["seqs"], c["new"], c["heads"], c["qd"])
    out = []
    for s in range(c["seqs"]):
        m = _past(c, s) + c["new"]
        k = kc[s, :m].double().view(m, c["kv_heads"], c["qd"])
        v = vc[s, :m].double().view(m, c["kv_heads"], c["vd"])
        out.append(_attend(q[s], k, v, _past(c, s), c["window"]))
    return torch.cat(out).view(c["seqs"] * c["new"], -1)


def _work_attention(c):
    pairs = cached = 0
    w = c["window"] or 1 << 30
    for s in range(c["seqs"]):
        past = _past(c, s)
        pairs += sum(min(past + i + 1, w) for i in range(c["new"]))
        cached += min(past + c["new"], w + c["new"] - 1)
    rows = c["seqs"] * c["new"]
    return {"bytes": 4 * ((cached * c["kv_heads"] + rows * c["heads"]) * (c["qd"] + c["vd"])),
            "flops": 2 * pairs * c["heads"] * (c["qd"] + c["vd"])}


# ------------------------------------------------------------------------ model

SHAPE = synth.model_shape("tiny_mixtral")


def _model_bytes(seed):
    """(name, format, shape, stored bytes) of every tensor of the model."""
    out = []
    for i, (name, dt, shape, fill) in enumerate(SHAPE.plan()):
        rows = int(np.prod(shape[:-1])) if len(shape) > 1 else 1
        if dt != F32:
            raw = _stored(seed, 1000 + i, dt, rows, shape[-1])
        else:
            v = _normal(seed, 1000 + i, shape, WEIGHT_STD)
            raw = (v + 1.0 if fill == "ones" else v).contiguous().view(torch.uint8).view(-1)
        out.append((name, dt, shape, raw))
    return out


def _tokens(c, seed):
    g = torch.Generator().manual_seed(int(seed) * 7919 + 5)
    return torch.randint(0, SHAPE.vocab, (c["seqs"], c["past"] + c["new"]), generator=g).tolist()


def _prepare_model(c, seed):
    parts = _model_bytes(seed)
    buf = torch.cat([p[3] for p in parts]).cpu().numpy()
    ck, at = HostCheckpoint(buf), 0
    for name, dt, shape, raw in parts:
        ck.add(name, HostTensor(dt, tuple(shape), buf[at:at + raw.numel()]), at)
        at += raw.numel()
    ctx = Context(0)
    spec = Spec.derive(SHAPE.config(), {n: t.shape for n, t in ck.items()})
    model = Model(ctx, spec, upload_store(ctx, ck), device=DEV)
    tokens = _tokens(c, seed)
    state = model.new_state(c["seqs"], c["past"] + c["new"])
    if c["past"]:
        model.forward([row[:c["past"]] for row in tokens], state)
    return {"model": model, "ctx": ctx, "state": state, "past": c["past"], "ids": [row[c["past"]:] for row in tokens]}


def _run_model(s):
    s["state"].pos = [s["past"]] * len(s["ids"])  # the same step again
    return s["model"].forward(s["ids"], s["state"])


def _exact_model(c, seed):
    raw = {n: (dt, shape, b) for n, dt, shape, b in _model_bytes(seed)}

    def mat(name):
        dt, shape, b = raw[name]
        if dt == F32:
            return b.view(torch.float32).view(shape).double()
        return _values(b, dt, shape[0], shape[1])

    def norm(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + SHAPE.eps) * w

    def turn(x, pos):  # rope on [n, heads, d]
        d = x.shape[2]
        inv = SHAPE.rope_theta ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
        ang = (pos[:, None] * inv)[:, None, :]
        a, b = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], 2)

    ids = torch.tensor(_tokens(c, seed), device=DEV)
    seqs, n = ids.shape
    pos = torch.arange(n, device=DEV, dtype=torch.float64)
    x = mat("model.embed_tokens.weight")[ids.view(-1)]
    for l in range(SHAPE.layers):
        p = "model.layers.%d." % l
        h = norm(x, mat(p + "input_layernorm.weight"))
        q, k, v = (h @ mat(p + "self_attn.%s_proj.weight" % m).T for m in "qkv")
        heads = []
        for s in range(seqs):
            r = slice(s * n, (s + 1) * n)
            qs = turn(q[r].view(n, SHAPE.heads, -1), pos)
            ks = turn(k[r].view(n, SHAPE.kv_heads, -1), pos)
            heads.append(_attend(qs, ks, v[r].view(n, SHAPE.kv_heads, -1), 0, 0).reshape(n, -1))
        x = x + torch.cat(heads) @ mat(p + "self_attn.o_proj.weight").T
        h = norm(x, mat(p + "post_attention_layernorm.weight"))
        b = p + "block_sparse_moe."
        score, sel = torch.softmax(h @ mat(b + "gate.weight").T, 1).topk(SHAPE.top_k, 1)
        w = score / score.sum(1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(SHAPE.n_experts):
            tok, slot = (sel == e).nonzero(as_tuple=True)
            gate, down, up = (mat(b + "experts.%d.w%d.weight" % (e, i)) for i in (1, 2, 3))
            y.index_add_(0, tok, _swiglu(h[tok], gate, up, down) * w[tok, slot][:, None])
        x = x + y
    last = norm(x.view(seqs, n, -1)[:, -1], mat("model.norm.weight"))
    return last @ mat("lm_head.weight").T


def _work_model(c):
    rows, H, m = c["seqs"] * c["new"], SHAPE.hidden, SHAPE
    proj = 2 * H * (m.heads + m.kv_heads) * m.head_dim
    expert = 3 * H * m.moe_inter
    hit = m.n_experts * (1.0 - (1.0 - m.top_k / m.n_experts) ** rows)
    pairs = c["seqs"] * sum(c["past"] + i + 1 for i in range(c["new"]))
    cached = c["seqs"] * (c["past"] + c["new"]) * 2 * m.kv_heads * m.head_dim * 4
    weights = _stored_bytes(m.dt, m.layers * proj + m.vocab * H + int(m.layers * hit) * expert)
    return {"bytes": int(weights + m.layers * (cached + 4 * m.n_experts * H) + c["seqs"] * m.vocab * 4),
            "flops": 2 * rows * m.layers * (proj + m.top_k * expert + m.n_experts * H)
                     + 4 * pairs * m.layers * m.heads * m.head_dim + 2 * c["seqs"] * m.vocab * H}


# -------------------------------------------------------------------- interface

_KINDS = {"layer": (_prepare_layer, _run_layer, _exact_layer, _work_layer),
          "linear": (_prepare_linear, _run_linear, _exact_linear, _work_linear),
          "attention": (_prepare_attention, _run_attention, _exact_attention, _work_attention),
          "model": (_prepare_model, _run_model, _exact_model, _work_model)}


def prepare(case, seed):
    state = _KINDS[case["kind"]][0](case, seed)
    state["run"] = _KINDS[case["kind"]][1]
    return state


def run(state):
    return state["run"](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    # 32-bit sums of products: about four times what the paths here differ by
    # from 64 bits (layers and projections 1e-7 to 5e-7, attention 3e-7 to
    # 7e-7, the model's logits 5e-7).
    return {"rel": 3e-6 if case["kind"] in ("attention", "model") else 2e-6}
