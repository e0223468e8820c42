"""Workloads of the Q8_0 embedding backend, from one projection of a short query
to a batch of texts through the whole backbone and the search over stored codes.

Every case goes through glypr_amd.ops, as an embedding service's program calls
it.  A case is a dict of plain values; `prepare` makes what the program has in
hand before the call (context, weights, inputs on the device), `run` is one
call, `exact` states the same result in 64 bits with plain torch.

Geometries: "base" is the 768-wide backbone (ffn 1152, 3 q heads on 1 kv head of
256), "released" the 512-wide one (ffn 2048, 4 q heads; sliding layers 2 kv heads
of 256, full-attention layers 1 kv head of 512, Per-Layer Embeddings and a
512 -> 768 embedding projection).  Whole-model cases run one layer of each kind
(sliding, full): a rounding that differs anywhere flips Q8_0 codes in every
projection behind it, so deeper stacks of random weights drift apart by more
than a tolerance could separate from a mistake.
"""
import math
import random

import numpy as np
import torch

from glypr_amd import ops

EPS = 1e-6
VOCAB = 32768
LAYER_TYPES = [0, 1]     # sliding, full attention
N_LAYERS = len(LAYER_TYPES)
WINDOW = 512
VARIANTS = {"exact": ops.INT8_EXACT, "bf16": ops.BF16_DEQUANT, "fma": ops.INT8_FMA}
GEOMETRY = {
    "base": dict(hidden=768, ffn=1152, n_heads=3, n_kv_heads=1, head_dim=256),
    "released": dict(hidden=512, ffn=2048, n_heads=4, n_kv_heads=2, head_dim=256,
                     full_head_dim=512, full_n_kv_heads=1, ple_dim=256, out_dim=768),
}
# (in, out) of the layers' projections: q|k|v, o, gate|up, down of both geometries
PROJECTIONS = [(768, 1280), (768, 768), (768, 2304), (1152, 768),
               (512, 2048), (1024, 512), (512, 3072), (2048, 512), (512, 768)]


def listed():
    return [
        # The o projection of a short query: the smallest call a program makes.
        dict(name="linear_query", kind="linear", m=17, k=768, n=768, norm=False, variant="exact"),
        # The q|k|v projection of one long document, norm and quantizer in front.
        dict(name="linear_doc", kind="linear", m=1213, k=768, n=1280, norm=True, variant="exact"),
        # The same projection over an indexing batch (32 x 512 tokens) for a caller
        # that takes bf16 arithmetic.
        dict(name="linear_bulk", kind="linear", m=16384, k=768, n=1280, norm=True, variant="bf16"),
        # The feed-forward block of a 512-token document, and of an indexing batch
        # of the released geometry.
        dict(name="mlp_doc", kind="mlp", m=512, hidden=768, ffn=1152, variant="exact"),
        dict(name="mlp_bulk", kind="mlp", m=8190, hidden=512, ffn=2048, variant="exact"),
        # A dense bf16 projection (files with F16 / BF16 tensors).
        dict(name="dense_doc", kind="dense", m=3001, k=1152, n=768),
        # Attention of one document: a sliding layer of the released geometry, and
        # its full layer at the longest context.
        dict(name="attn_sliding", kind="attention", t=1777, n_heads=4, n_kv_heads=2, head_dim=256,
             window=WINDOW),
        dict(name="attn_full", kind="attention", t=8192, n_heads=4, n_kv_heads=1, head_dim=512,
             window=0),
        # Search: a service's query batch against stored int8 codes, and one query
        # against a large binary index.
        dict(name="search_int8", kind="search", codec="int8", na=24, nb=200003, dim=768),
        dict(name="search_binary", kind="search", codec="binary", na=1, nb=1000000, dim=256),
        # One document through the released backbone.
        dict(name="embed_doc", kind="embed", geometry="released", t=333, variant="exact"),
        # A batch of short and long texts through the base backbone.
        dict(name="embed_batch", kind="batch", geometry="base", n_seqs=40, shortest=5, longest=500,
             lens_seed=1, variant="exact"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "dense", "attention", "attention", "search",
                       "search", "embed", "batch"])
    if kind == "linear":
        if rng.random() < 0.75:
            k, n = rng.choice(PROJECTIONS)
        else:   # any weight of a Q8_0 file
            k, n = 32 * rng.randint(8, 64), rng.randint(100, 3000)
        return dict(kind=kind, m=_log_int(rng, 1, 16384), k=k, n=n, norm=rng.random() < 0.5,
                    variant=rng.choice(["exact", "exact", "fma", "bf16"]))
    if kind == "mlp":
        hidden, ffn = rng.choice([(768, 1152), (512, 2048)])
        return dict(kind=kind, m=_log_int(rng, 1, 12000), hidden=hidden, ffn=ffn,
                    variant=rng.choice(["exact", "exact", "fma", "bf16"]))
    if kind == "dense":
        k, n = rng.choice(PROJECTIONS)
        return dict(kind=kind, m=_log_int(rng, 1, 16384), k=k, n=n)
    if kind == "attention":
        n_heads, n_kv_heads, head_dim, window = rng.choice(
            [(3, 1, 256, 0), (3, 1, 256, WINDOW), (4, 2, 256, WINDOW), (4, 1, 512, 0)])
        return dict(kind=kind, t=_log_int(rng, 8, 8192), n_heads=n_heads, n_kv_heads=n_kv_heads,
                    head_dim=head_dim, window=window)
    if kind == "search":
        dim = rng.choice([128, 256, 512, 768])
        na = _log_int(rng, 1, 64)
        return dict(kind=kind, codec=rng.choice(["int8", "binary"]), na=na,
                    nb=_log_int(rng, 1000, 6000000 // max(na, 24)), dim=dim)
    if kind == "embed":
        return dict(kind=kind, geometry=rng.choice(["base", "released"]), t=_log_int(rng, 4, 1500),
                    variant=rng.choice(["exact", "exact", "fma"]))
    shortest = _log_int(rng, 3, 40)
    return dict(kind="batch", geometry=rng.choice(["base", "released"]), n_seqs=rng.randint(2, 24),
                shortest=shortest, longest=_log_int(rng, shortest + 1, 400),
                lens_seed=rng.randrange(1 << 20), variant=rng.choice(["exact", "exact", "fma"]))


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _round_away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _q8(x):
    """BlockQ8_0::from_float over the last axis: (codes, f16 scales) per 32 values."""
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    return _round_away(b * inv[..., None]).clamp(-128, 127).to(torch.int8), d.half()


def _deq64(codes, d):
    return (codes.double() * d.double()[..., None]).flatten(-2)


def _q8_64(x):
    """The value the Q8_0 operand of activations x has, in 64 bits."""
    return _deq64(*_q8(x))


def _q8_tensor(g, n, k, sigma=0.02):
    """A Q8_0 weight: (GGUF blocks on the host, its value in 64 bits on demand)."""
    codes, d = _q8(_normal(g, n, k) * sigma)
    blocks = torch.cat([d[..., None].view(torch.uint8), codes.view(torch.uint8)], dim=-1)
    return blocks.reshape(n, -1).cpu().numpy(), (codes, d)


def _norm_weight(g, n, scale=1.0):
    return (1 + 0.1 * _normal(g, n)) * scale


def _rope(t, head_dim, theta):
    i = torch.arange(head_dim // 2, dtype=torch.float64)
    inv = (1.0 / theta ** (2 * i / head_dim)).float()
    f = torch.arange(t, dtype=torch.float32)[:, None] * inv[None, :]
    f = torch.cat([f, f], 1)
    return f.cos().cuda(), f.sin().cuda()


def _lens(case):
    r = random.Random(case["lens_seed"])
    return [_log_int(r, case["shortest"], case["longest"]) for _ in range(case["n_seqs"])]


def _linear_inputs(case, seed):
    g = _gen(seed)
    blocks, w = _q8_tensor(g, case["n"], case["k"])
    return blocks, w, _normal(g, case["m"], case["k"]), _norm_weight(g, case["k"])


def _mlp_inputs(case, seed):
    g = _gen(seed)
    H, F = case["hidden"], case["ffn"]
    gate, up, down = _q8_tensor(g, F, H), _q8_tensor(g, F, H), _q8_tensor(g, H, F)
    return gate, up, down, _normal(g, case["m"], H), _norm_weight(g, H)


def _dense_inputs(case, seed):
    g = _gen(seed)
    w = (_normal(g, case["n"], case["k"]) * 0.02).bfloat16()
    return w, _normal(g, case["m"], case["k"])


def _attention_inputs(case, seed):
    g = _gen(seed)
    hd = case["head_dim"]
    qkv = _normal(g, case["t"], (case["n_heads"] + 2 * case["n_kv_heads"]) * hd) * 0.7
    # the q/k norms carry the attention scale (there is no 1/sqrt(head_dim))
    qn, kn = _norm_weight(g, hd, 0.25), _norm_weight(g, hd, 0.25)
    cos, sin = _rope(case["t"], hd, 10000.0 if case["window"] else 1e6)
    return qkv, qn, kn, cos, sin


def _unit_rows(g, n, dim):
    x = _normal(g, n, dim)
    return x / x.norm(dim=1, keepdim=True)


def _int8_codes(x):
    return _round_away(x * 127.0).clamp(-127, 127).to(torch.int8)


def _bits(x):
    """int64 words whose bit i is x[64 w + i] > 0."""
    b = (x > 0).reshape(x.shape[0], -1, 64)
    shift = torch.arange(64, device="cuda", dtype=torch.int64)
    return (b.to(torch.int64) << shift).sum(-1)


def _search_inputs(case, seed):
    g = _gen(seed)
    q = _unit_rows(g, case["na"], case["dim"])
    encode = _int8_codes if case["codec"] == "int8" else _bits
    step = 1 << 16
    db = [encode(_unit_rows(g, min(step, case["nb"] - i), case["dim"]))
          for i in range(0, case["nb"], step)]
    return q, torch.cat(db)


def _model_tensors(case, seed):
    """{GGUF name: (host array, rows, cols, is Q8_0)} and the same for `exact`."""
    g = _gen(seed)
    c = GEOMETRY[case["geometry"]]
    H, F, nq = c["hidden"], c["ffn"], c["n_heads"]
    host, dev = {}, {}

    def q8(name, n, k, sigma=0.02):
        blocks, dev[name] = _q8_tensor(g, n, k, sigma)
        host[name] = (blocks, n, k, True)

    def f32(name, v):
        dev[name] = v
        host[name] = (v.cpu().numpy(), 1, v.numel(), False)

    q8("token_embd.weight", VOCAB, H)
    f32("output_norm.weight", _norm_weight(g, H))
    P = c.get("ple_dim", 0)
    if P:
        q8("per_layer_model_proj.weight", N_LAYERS * P, H, 0.05)
        f32("per_layer_proj_norm.weight", _norm_weight(g, P))
    if c.get("out_dim"):
        q8("output.weight", c["out_dim"], H, 0.05)
    for i in range(N_LAYERS):
        hd, nkv = _layer_heads(c, i)
        for name, n, k in [("attn_q", nq * hd, H), ("attn_k", nkv * hd, H), ("attn_v", nkv * hd, H),
                           ("attn_output", H, nq * hd), ("ffn_gate", F, H), ("ffn_up", F, H),
                           ("ffn_down", H, F)]:
            q8(f"blk.{i}.{name}.weight", n, k)
        for name in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
            f32(f"blk.{i}.{name}.weight", _norm_weight(g, H))
        for name in ("attn_q_norm", "attn_k_norm"):
            f32(f"blk.{i}.{name}.weight", _norm_weight(g, hd, 0.25))
        if P:
            q8(f"blk.{i}.inp_gate.weight", P, H, 0.05)
            q8(f"blk.{i}.proj.weight", H, P, 0.05)
            f32(f"blk.{i}.post_norm.weight", _norm_weight(g, H))
            f32(f"blk.{i}.layer_output_scale.weight",
                0.5 + 0.5 * torch.rand(1, generator=g, device="cuda"))
    return host, dev


def _layer_heads(c, i):
    if not LAYER_TYPES[i]:
        return c["head_dim"], c["n_kv_heads"]
    return c.get("full_head_dim", c["head_dim"]), c.get("full_n_kv_heads", c["n_kv_heads"])


def _ids(case, seed):
    r = np.random.default_rng(seed)
    lens = [case["t"]] if case["kind"] == "embed" else _lens(case)
    return [r.integers(0, VOCAB, n).astype(np.uint32) for n in lens]


def prepare(case, seed):
    kind = case["kind"]
    ctx = ops.Context(0)
    st = dict(case=case, ctx=ctx)
    if kind == "linear":
        blocks, _, st["x"], nw = _linear_inputs(case, seed)
        st["w"] = ops.Q8Weight.from_gguf(ctx, blocks, case["n"], case["k"])
        st["norm"] = nw if case["norm"] else None
        if case["m"] > 8320:
            ctx.reserve(case["m"])
    elif kind == "mlp":
        gate, up, down, st["x"], st["norm"] = _mlp_inputs(case, seed)
        H, F = case["hidden"], case["ffn"]
        st["gate_up"] = ops.Q8Weight.from_gguf(ctx, np.concatenate([gate[0], up[0]]), 2 * F, H)
        st["down"] = ops.Q8Weight.from_gguf(ctx, down[0], H, F)
        if case["m"] > 8320:
            ctx.reserve(case["m"])
    elif kind == "dense":
        w, st["x"] = _dense_inputs(case, seed)
        st["w"] = ops.BF16Weight.from_bf16(ctx, w.view(torch.int16).cpu().numpy().view(np.uint16))
        if case["m"] > 8320:
            ctx.reserve(case["m"])
    elif kind == "attention":
        st["qkv"], st["qn"], st["kn"], st["cos"], st["sin"] = _attention_inputs(case, seed)
    elif kind == "search":
        st["q"], st["db"] = _search_inputs(case, seed)
    else:
        host, _ = _model_tensors(case, seed)
        ids = _ids(case, seed)
        rows = sum(-(-len(s) // 64) * 64 for s in ids)
        m = ops.Model(ctx, layer_types=LAYER_TYPES, n_layers=N_LAYERS, vocab=VOCAB, sliding_window=WINDOW,
                      max_seq_len=2048, max_batch_tokens=max(2048, rows),
                      **GEOMETRY[case["geometry"]])
        for name, (data, r, c, q8) in host.items():
            m.set_tensor(name, data, r, c, q8)
        m.finalize()
        m.set_variant(VARIANTS[case["variant"]])
        st["model"], st["ids"] = m, ids
        if kind == "embed":
            c = GEOMETRY[case["geometry"]]
            st["hidden"] = torch.empty(case["t"], c.get("out_dim") or c["hidden"], device="cuda")
    torch.cuda.synchronize()
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "linear":
        v = VARIANTS[case["variant"]]
        if st["norm"] is None:
            return ops.q8_0_matmul(ctx, st["w"], st["x"], v)
        return ops.rmsnorm_q8_0_matmul(ctx, st["w"], st["x"], st["norm"], EPS, v)
    if kind == "mlp":
        return ops.rmsnorm_mlp(ctx, st["gate_up"], st["down"], st["x"], st["norm"], EPS,
                               VARIANTS[case["variant"]])
    if kind == "dense":
        return ops.bf16_matmul(ctx, st["w"], st["x"])
    if kind == "attention":
        return ops.attention(ctx, st["qkv"], st["qn"], st["kn"], EPS, st["cos"], st["sin"],
                             case["n_heads"], case["n_kv_heads"], case["head_dim"], case["window"])
    if kind == "search":
        if case["codec"] == "int8":
            codes = ops.quantize_int8(ctx, st["q"])
            return {"codes": codes, "scores": ops.int8_cosine(ctx, codes, st["db"])}
        codes = ops.quantize_binary(ctx, st["q"])
        return {"codes": codes, "scores": ops.binary_cosine(ctx, codes, st["db"])}
    if kind == "embed":
        out = st["model"].embed(st["ids"][0], trunc=256, hidden=st["hidden"])
        return {"embedding": out, "hidden": st["hidden"]}
    return st["model"].embed_batch(st["ids"], trunc=256)


# ---- what a pass cannot do without ------------------------------------------

def _pairs(t, window):
    """Query-key pairs of one head."""
    if not window or t <= window:
        return t * t
    return t * (2 * window + 1) - window * (window + 1)


def work(case):
    kind = case["kind"]
    q8 = 34 / 32
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4 * m * (k + n) + q8 * n * k, flops=2 * m * n * k)
    if kind == "mlp":
        m, H, F = case["m"], case["hidden"], case["ffn"]
        return dict(bytes=8 * m * H + q8 * 3 * F * H, flops=6 * m * F * H)
    if kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4 * m * (k + n) + 2 * n * k, flops=2 * m * n * k)
    if kind == "attention":
        t, nq, nkv, hd = (case[x] for x in ("t", "n_heads", "n_kv_heads", "head_dim"))
        return dict(bytes=4 * t * hd * (2 * nq + 2 * nkv + 2),
                    flops=4 * _pairs(t, case["window"]) * nq * hd)
    if kind == "search":
        na, nb, dim = case["na"], case["nb"], case["dim"]
        if case["codec"] == "int8":
            return dict(bytes=nb * dim + 4 * na * nb + 5 * na * dim, flops=2 * na * nb * dim)
        return dict(bytes=nb * dim / 8 + 4 * na * nb + 4 * na * dim, flops=0)
    c = GEOMETRY[case["geometry"]]
    lens = [case["t"]] if kind == "embed" else _lens(case)
    rows, H, F, nq = sum(lens), c["hidden"], c["ffn"], c["n_heads"]
    P, D = c.get("ple_dim", 0), c.get("out_dim", 0)
    params, attn = N_LAYERS * P * H + D * H, 0
    for i in range(N_LAYERS):
        hd, nkv = _layer_heads(c, i)
        params += H * hd * (2 * nq + 2 * nkv) + 3 * H * F + 2 * H * P
        attn += sum(4 * _pairs(t, 0 if LAYER_TYPES[i] else WINDOW) * nq * hd for t in lens)
    out = rows * (D or H) if kind == "embed" else 0
    return dict(bytes=q8 * (params + rows * H) + 4 * (out + 256 * len(lens)),
                flops=2 * rows * params + attn)


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "mlp"):
        # INT8_EXACT is bit-identical by contract.  INT8_FMA: sums of 32-bit terms in
        # another order, and behind a norm or inside the feed-forward block Q8_0
        # codes that sit on a rounding boundary.  bf16: operands of 8 bits.
        if case["variant"] == "exact":
            return "exact"
        if case["variant"] == "bf16":
            return {"rel": 1e-2}
        if kind == "mlp":
            return {"rel": 1e-3, "max": 0.1}
        return {"rel": 2e-4 if case["norm"] else 1e-5}
    if kind == "dense":
        return {"rel": 1e-5}    # the same bf16 operands, 32-bit sums in another order
    if kind == "attention":
        return {"rel": 2e-3}    # f16 operands and probabilities, 32-bit sums
    if kind == "search":
        return {"rel": 1e-6}    # exact integer sums, one 32-bit division
    # f16 attention operands, then Q8_0 roundings that flip in every layer behind
    return {"rel": 3e-2, "max": 0.5}


# ---- the same in 64 bits ----------------------------------------------------

def _rms64(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(0.7978846 * (x + 0.044715 * x ** 3)))


def _linear64(x, w, quantized=True):
    return (_q8_64(x) if quantized else x) @ _deq64(*w).T


def _rotate64(x, cos, sin):     # x [t, heads, hd]
    half = x.shape[-1] // 2
    rot = torch.cat([-x[..., half:], x[..., :half]], -1)
    return x * cos.double()[:, None] + rot * sin.double()[:, None]


def _attention64(qkv, qn, kn, cos, sin, n_heads, n_kv_heads, hd, window):
    t = qkv.shape[0]
    q, k, v = qkv.double().split([n_heads * hd, n_kv_heads * hd, n_kv_heads * hd], 1)
    q = _rotate64(_rms64(q.reshape(t, n_heads, hd), qn), cos, sin)
    k = _rotate64(_rms64(k.reshape(t, n_kv_heads, hd), kn), cos, sin)
    v = _rms64(v.reshape(t, n_kv_heads, hd))
    out = torch.empty(t, n_heads, hd, dtype=torch.float64, device=qkv.device)
    pos = torch.arange(t, device=qkv.device)
    for h in range(n_heads):
        g = h // (n_heads // n_kv_heads)
        kh, vh = k[:, g].contiguous(), v[:, g].contiguous()
        for i in range(0, t, 1024):
            s = q[i:i + 1024, h].contiguous() @ kh.T
            if window and t > window:
                s.masked_fill_((pos[i:i + 1024, None] - pos[None]).abs() > window, -math.inf)
            out[i:i + 1024, h] = torch.softmax(s, -1) @ vh
    return out.reshape(t, n_heads * hd)


def _forward64(geometry, w, ids):
    c = GEOMETRY[geometry]
    H, nq, t = c["hidden"], c["n_heads"], len(ids)
    codes, d = w["token_embd.weight"]
    at = torch.from_numpy(ids.astype(np.int64)).cuda()
    h = _deq64(codes[at], d[at]) * float(np.float32(math.sqrt(H)))
    P = c.get("ple_dim", 0)
    if P:
        ple = _linear64(h, w["per_layer_model_proj.weight"]) * H ** -0.5
        ple = _rms64(ple.reshape(t, N_LAYERS, P), w["per_layer_proj_norm.weight"])
    for i in range(N_LAYERS):
        L = {n[len(f"blk.{i}."):-len(".weight")]: v for n, v in w.items()
             if n.startswith(f"blk.{i}.")}
        full = LAYER_TYPES[i]
        hd, nkv = _layer_heads(c, i)
        x = _rms64(h, L["attn_norm"])
        qkv = torch.cat([_linear64(x, L[n]) for n in ("attn_q", "attn_k", "attn_v")], 1)
        cos, sin = _rope(t, hd, 1e6 if full else 10000.0)
        a = _attention64(qkv, L["attn_q_norm"], L["attn_k_norm"], cos, sin, nq, nkv, hd,
                         0 if full else WINDOW)
        h = h + _rms64(_linear64(a, L["attn_output"]), L["post_attention_norm"])
        x = _rms64(h, L["ffn_norm"])
        f = _gelu64(_linear64(x, L["ffn_gate"])) * _linear64(x, L["ffn_up"])
        h = h + _rms64(_linear64(f, L["ffn_down"]), L["post_ffw_norm"])
        if P:
            p = _gelu64(_linear64(h, L["inp_gate"])) * ple[:, i]
            h = (h + _rms64(_linear64(p, L["proj"]), L["post_norm"])) * \
                L["layer_output_scale"].double()
    states = _rms64(h, w["output_norm.weight"])
    if c.get("out_dim"):
        states = _linear64(states, w["output.weight"])
    e = states.mean(0)
    e = (e / e.norm())[:256]
    return e / e.norm(), states


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        _, w, x, nw = _linear_inputs(case, seed)
        x = x.double()
        if case["norm"]:
            x = _rms64(x, nw)
        return _linear64(x, w, case["variant"] != "bf16")
    if kind == "mlp":
        gate, up, down, x, nw = _mlp_inputs(case, seed)
        quantized = case["variant"] != "bf16"
        x = _rms64(x.double(), nw)
        h = _gelu64(_linear64(x, gate[1], quantized)) * _linear64(x, up[1], quantized)
        return _linear64(h, down[1], quantized)
    if kind == "dense":
        w, x = _dense_inputs(case, seed)
        return x.double() @ w.double().T
    if kind == "attention":
        return _attention64(*_attention_inputs(case, seed), case["n_heads"], case["n_kv_heads"],
                            case["head_dim"], case["window"])
    if kind == "search":
        q, db = _search_inputs(case, seed)
        if case["codec"] == "int8":
            a = _int8_codes(q).double()
            out = torch.empty(a.shape[0], db.shape[0], dtype=torch.float64, device="cuda")
            for i in range(0, db.shape[0], 1 << 15):
                b = db[i:i + (1 << 15)].double()
                out[:, i:i + (1 << 15)] = (a @ b.T) / (a.norm(dim=1)[:, None] * b.norm(dim=1))
            return {"codes": None, "scores": out.clamp(-1, 1)}
        a = _bits(q)
        ones = torch.tensor([bin(i).count("1") for i in range(256)], device="cuda")
        out = torch.empty(a.shape[0], db.shape[0], dtype=torch.float64, device="cuda")
        for i in range(a.shape[0]):
            x = (a[i] ^ db).view(torch.uint8)
            for j in range(0, db.shape[0], 1 << 18):
                h = ones[x[j:j + (1 << 18)].long()].sum(1)
                out[i, j:j + (1 << 18)] = torch.cos(math.pi * h.double() / case["dim"])
        return {"codes": None, "scores": out}
    _, w = _model_tensors(case, seed)
    got = [_forward64(case["geometry"], w, ids) for ids in _ids(case, seed)]
    if kind == "embed":
        return {"embedding": got[0][0], "hidden": got[0][1]}
    return torch.stack([e for e, _ in got])
