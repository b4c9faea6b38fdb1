"""The work whose speed is measured: model steps as the serving engine makes them, through the models' own ``forward``, and
the mixture-of-experts feed-forward through :mod:`chronos.ops.hybrid`.

A case is a dict of sizes.  Kinds:

* ``llama_prefill`` / ``llama_decode``: one prefill step of several prompts / one graph-captured decode step, Llama-3 8B
  widths, four layers and the whole vocabulary (a layer is a layer: the other 28 repeat these);
* ``llama_long``: a decode step over long contexts with an fp8 KV cache;
* ``hybrid_prefill`` / ``hybrid_decode``: the same two steps of a hybrid design at the sizes of
  ``chronos.utils.design_bench`` (four layers), its feed-forwards dense: a router's choice between near-equal experts
  turns on the last bit of its input, so whole models with routers have no result that two correct programs share;
* ``moe``: router and experts by themselves, on given activations.

Decode steps are replayed from a captured graph and prefill steps run eagerly, as the engine runs them.  Outputs are the
logits and everything the step writes: pages of keys and values, recurrent states, convolution histories.
"""
from __future__ import annotations

import dataclasses
import math
import random

import torch

from chronos import ops
from chronos.models import kalesun, llama, vogerax, zokunex
from chronos.models.hybrid import HybridDecoder
from chronos.models.llama import StepBatch
from chronos.ops import hybrid as hops
from chronos.utils import design_bench as db

BS = 16          # cache page, tokens (the engine's default)
LAYERS = 4
F64 = torch.float64
DESIGNS = {"zokunex": (zokunex, db.zokunex_config, db.SIZES), "kalesun": (kalesun, db.kalesun_config, db.KALESUN_SIZES),
           "vogerax": (vogerax, db.vogerax_config, db.VOGERAX_SIZES)}


def listed():
    return [
        # one sensor's verdict being written: one row, a chain's prompt and part of the reply behind it
        dict(name="llama_decode_1", kind="llama_decode", rows=1, ctx=140),
        # 1024 sensor streams decoding together (the headline benchmark's wave)
        dict(name="llama_decode_1024", kind="llama_decode", rows=1024, ctx=120),
        # prompts of newly arrived chains, one prefill step
        dict(name="llama_prefill_64", kind="llama_prefill", seqs=64, tokens=93),
        # two investigations over a 128k-token history each, fp8 pages
        dict(name="llama_long_128k", kind="llama_long", rows=2, ctx=131000),
        # hybrid designs: the prompt step of four 2048-token histories, at the three widths
        dict(name="zokunex_prefill_2k", kind="hybrid_prefill", design="zokunex", size="2k", seqs=4, tokens=2048, ragged=False),
        dict(name="vogerax_prefill_1k", kind="hybrid_prefill", design="vogerax", size="1k", seqs=4, tokens=2048, ragged=False),
        dict(name="kalesun_prefill_4k", kind="hybrid_prefill", design="kalesun", size="4k", seqs=4, tokens=2048, ragged=False),
        # ... and of short chains of unequal length, odd sizes
        dict(name="kalesun_prefill_chains", kind="hybrid_prefill", design="kalesun", size="1k", seqs=21, tokens=117, ragged=True),
        # their decode steps: a batch in the middle of its replies, one stream alone
        dict(name="zokunex_decode_64", kind="hybrid_decode", design="zokunex", size="4k", rows=64, ctx=2048),
        dict(name="kalesun_decode_1", kind="hybrid_decode", design="kalesun", size="1k", rows=1, ctx=700),
        # experts: a prompt step's tokens through gated experts, a decode batch's through plain ones
        dict(name="moe_glu_8192", kind="moe", form="glu", size="2k", tokens=8192),
        dict(name="moe_gelu_64", kind="moe", form="gelu", size="4k", tokens=64),
    ]


def draw(rng):
    log = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    kind = rng.choice(["llama_decode", "llama_prefill", "llama_long", "hybrid_prefill", "hybrid_prefill", "hybrid_decode",
                       "hybrid_decode", "moe"])
    if kind == "llama_decode":
        return dict(kind=kind, rows=log(1, 1024), ctx=log(40, 500))
    if kind == "llama_prefill":
        seqs = log(1, 64)
        return dict(kind=kind, seqs=seqs, tokens=log(20, min(2048, 6000 // seqs)))
    if kind == "llama_long":
        rows = log(1, 8)
        return dict(kind=kind, rows=rows, ctx=log(4096, 262000 // rows))
    if kind == "hybrid_prefill":
        seqs = log(1, 32)
        return dict(kind=kind, design=rng.choice(sorted(DESIGNS)), size=rng.choice(["1k", "2k", "4k"]), seqs=seqs,
                    tokens=log(20, min(4000, 8000 // seqs)), ragged=True)
    if kind == "hybrid_decode":
        return dict(kind=kind, design=rng.choice(["kalesun", "zokunex"]), size=rng.choice(["1k", "2k", "4k"]), rows=log(1, 64),
                    ctx=log(50, 3000))
    return dict(kind=kind, form=rng.choice(["glu", "gelu"]), size=rng.choice(["1k", "2k", "4k"]), tokens=log(1, 8192))


# ---- sizes ---------------------------------------------------------------------------------------------------------


def _spread(case, n, mean, least=1):
    """n lengths around a mean, the same for every seed."""
    r = random.Random("%d %d" % (n, mean))
    return [max(least, int(round(mean * r.uniform(0.6, 1.4)))) for _ in range(n)]


def _lens(case):
    """Tokens per sequence: the prompt's in a prefill step, those already cached in a decode step."""
    if case["kind"] in ("llama_prefill", "hybrid_prefill"):
        if case["kind"] == "hybrid_prefill" and not case["ragged"]:
            return [case["tokens"]] * case["seqs"]
        return _spread(case, case["seqs"], case["tokens"])
    if case["kind"] == "llama_long":
        return [case["ctx"] - 37 * i for i in range(case["rows"])]
    return _spread(case, case["rows"], case["ctx"])


def _llama_config(case):
    top = max(_lens(case)) + 2
    return dataclasses.replace(llama.get_config("llama3-8b"), num_layers=LAYERS, max_position=max(8192, top))


def _hybrid_dict(case):
    _, make, sizes = DESIGNS[case["design"]]
    size = sizes[case["size"]]
    cfg = make(size)
    for l in cfg["layers"]:
        if l["mlp"]["kind"] == "moe":
            l["mlp"] = dict(kind="dense", ff=size["ff"], limit=7.0)
    return cfg


def _hybrid_config(case):
    return DESIGNS[case["design"]][0].config_from_dict(_hybrid_dict(case), max_position=8192)


def _moe_sizes(case):
    """(width, experts with weights, identity experts, chosen, expert size)"""
    if case["form"] == "glu":
        s = db.KALESUN_SIZES[case["size"]]
        return (s["width"], s["moe"][0], 0, s["moe"][1], s["moe"][2])
    s = db.SIZES[case["size"]]
    return (s["width"], s["moe"][0], s["moe"][1], s["moe"][2], s["moe"][3])


# ---- inputs --------------------------------------------------------------------------------------------------------


def _dev():
    ops.load()
    hops.load()
    ops.device_init()
    return torch.device("cuda:0")


def _gen(dev, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return g


def _hybrid_tensors(cfg, mod, dev, seed):
    """Checkpoint-named random weights in bfloat16, scaled like the designs' own random weights.  The keys of the recurrent
    layers lean towards their queries: a sequence's first read-out, (k . q) v scaled to unit size, would otherwise be a
    random sign times its value, which no two programs share."""
    g, out = _gen(dev, seed), {}
    for name, shape in mod.tensor_shapes(cfg).items():
        leaf = name.rsplit(".", 1)[-1]
        if len(shape) == 0:
            t = torch.rand((), generator=g, device=dev) * 0.5 + 0.2
        elif len(shape) == 1:
            t = torch.randn(shape, generator=g, device=dev) * 0.1
            t += 0.5 if leaf in ("norm1b", "norm2b") else 1.0 if "norm" in name or leaf == "out" else 0.0
            t += 2.0 if name.endswith(("a2.b", "f.b")) else 0.0
        else:
            t = torch.randn(shape, generator=g, device=dev) * (0.5 if leaf == "conv" else shape[1] ** -0.5)
            q = out.get(name[:-1] + "q")
            if leaf == "k" and q.shape == t.shape:
                t = 0.6 * q.float() + 0.8 * t
        out[name] = t.to(torch.bfloat16)
    return out


def _packed(cfg, mod, tensors, dev):
    """The checkpoint's tensors laid out for the kernels; its few-number tensors come from host memory, as a file's do."""
    return mod.pack_weights(cfg, {n: t.cpu() if t.dim() < 2 else t for n, t in tensors.items()}, dev, torch.bfloat16)


def _pages(lens):
    """Page lists of the sequences, every page its own, page 0 left to the engine's scratch; pages in all."""
    out, at = [], 1
    for n in lens:
        k = -(-n // BS)
        out.append(list(range(at, at + k)))
        at += k
    return out, at


def _decode_batch(lens, vocab, hkv, dev, seed, slots):
    """Decode rows as the engine holds them: row i is sequence i, its next token at position lens[i]."""
    rows = len(lens)
    bts, nb = _pages([n + 1 for n in lens])
    i32 = dict(dtype=torch.int32, device=dev)
    mb = max(len(b) for b in bts)
    bt = torch.tensor([b + [0] * (mb - len(b)) for b in bts], **i32)
    pos, ar = torch.tensor(lens, **i32), torch.arange(rows + 1, **i32)
    ids = torch.randint(0, vocab, (rows,), generator=_gen(dev, seed + 1), device=dev).int()
    sb = StepBatch(ids, pos, ar[:rows], bt, ar, pos + 1, torch.arange(rows, device=dev), None, rows, 1,
                   ops.pick_nsplit(rows * hkv, max(lens) + 1), slots=ar[:rows].clone() if slots else None, max_q=1)
    return sb, nb


def _captured(step, keep):
    """One decode step captured as the engine captures its bursts; the warm-up's effect on the state is undone."""
    kept = [t.clone() for t in keep]
    step()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = step()
    for t, k in zip(keep, kept):
        t.copy_(k)
    torch.cuda.synchronize()
    return g, out


def _prepare_llama(case, seed, dev):
    cfg = _llama_config(case)
    lens = _lens(case)
    model = llama.LlamaModel(cfg, llama.random_weights(cfg, None, dev, seed), None, dev, cfg.max_position)
    if case["kind"] == "llama_prefill":
        bts, nb = _pages(lens)
        kv = model.make_cache(nb, BS, len(lens))
        ids = torch.randint(0, cfg.vocab_size, (sum(lens),), generator=_gen(dev, seed + 1), device=dev).tolist()
        at = [sum(lens[:i]) for i in range(len(lens) + 1)]
        sb = model.prefill_batch([ids[a:b] for a, b in zip(at, at[1:])], [0] * len(lens), bts, nqt=8)
        return dict(model=model, kv=kv, sb=sb, call=lambda: model.forward(sb, kv), out=[kv.buf])
    sb, nb = _decode_batch(lens, cfg.vocab_size, model.hkv, dev, seed, False)
    kv = model.make_cache(nb, BS, len(lens), "fp8" if case["kind"] == "llama_long" else "bf16")
    g = _gen(dev, seed + 2)
    for l in range(LAYERS):
        for side in range(2):
            t = torch.empty(kv.buf[l, side].shape, device=dev, dtype=torch.bfloat16).normal_(0.0, 0.7, generator=g)
            kv.buf[l, side].copy_(t.to(torch.float8_e4m3fn).view(torch.uint8) if kv.buf.dtype == torch.uint8 else t)
    # the new tokens' pages are written by the step itself: no state that its repetition changes
    graph, logits = _captured(lambda: model.forward(sb, kv), [kv.buf])
    return dict(model=model, kv=kv, sb=sb, graph=graph, logits=logits, out=[kv.buf])


def _prepare_hybrid(case, seed, dev):
    mod = DESIGNS[case["design"]][0]
    cfg, lens = _hybrid_config(case), _lens(case)
    model = HybridDecoder(cfg, _packed(cfg, mod, _hybrid_tensors(cfg, mod, dev, seed), dev), dev, 8192, torch.bfloat16)
    if case["kind"] == "hybrid_prefill":
        bts, nb = _pages(lens)
        cache = model.make_cache(nb, BS, len(lens))
        ids = torch.randint(0, cfg.vocab_size, (sum(lens),), generator=_gen(dev, seed + 1), device=dev).tolist()
        at = [sum(lens[:i]) for i in range(len(lens) + 1)]
        sb = model.prefill_batch([ids[a:b] for a, b in zip(at, at[1:])], [0] * len(lens), bts, list(range(len(lens))), nqt=8)
        return dict(model=model, kv=cache, sb=sb, call=lambda: model.forward(sb, cache), out=_cache_tensors(cache))
    sb, nb = _decode_batch(lens, cfg.vocab_size, model.hkv, dev, seed, True)
    cache = model.make_cache(nb, BS, len(lens))
    g = _gen(dev, seed + 2)
    for name, scale in (("lat", 1.0), ("kc", 1.0), ("vc", 0.7), ("hist", 0.7), ("S", 0.3), ("n", 0.5), ("m", 0.5)):
        for t in getattr(cache, name).values():
            t.normal_(0.0, scale, generator=g)
    state = [t for name in ("S", "n", "m", "hist") for t in getattr(cache, name).values()]
    graph, logits = _captured(lambda: model.forward(sb, cache), state)
    return dict(model=model, kv=cache, sb=sb, graph=graph, logits=logits, out=_cache_tensors(cache))


def _cache_tensors(cache):
    return [t for name in ("S", "n", "m", "lat", "kc", "vc", "kp", "vp", "hist") for t in getattr(cache, name).values()]


def _moe_inputs(case, seed, dev):
    d, ne, ni, top, ff = _moe_sizes(case)
    g = _gen(dev, seed)
    rnd = lambda *s, sc=1.0, dt=torch.bfloat16: torch.empty(*s, device=dev, dtype=torch.float32).normal_(0.0, sc, generator=g).to(dt)  # noqa: E731
    rows = 2 * ff if case["form"] == "glu" else ff
    return dict(h=rnd(case["tokens"], d), w_r=rnd(ne + ni, d, sc=2.0 * d ** -0.5), b=rnd(ne + ni, sc=0.01, dt=torch.float32),
                w_up=rnd(ne, rows, d, sc=d ** -0.5), w_down=rnd(ne, d, ff, sc=ff ** -0.5))


def _prepare_moe(case, seed, dev):
    t = _moe_inputs(case, seed, dev)
    top, ff = _moe_sizes(case)[3:]
    bf = torch.bfloat16
    if case["form"] == "glu":
        # a model keeps its gate and up rows in the order of the grouped matrix-core kernel
        w_gu = t["w_up"][:, hops.moe_glu_row_order(ff).to(dev)].contiguous()

        def call():
            idx, wt = hops.moe_route_topk(t["h"], t["w_r"], t["b"], top)
            return dict(idx=idx, wt=wt, y=hops.moe_glu_ffn(t["h"], idx, wt, w_gu, t["w_down"], 7.0, 1.702, 1.0, bf, True))
    else:
        def call():
            idx, wt = hops.moe_route(t["h"], t["w_r"], t["b"], top)
            return dict(idx=idx, wt=wt, y=hops.moe_ffn(t["h"], idx, wt, t["w_up"], t["w_down"], hops.ACT_GELU, bf))
    return dict(call=call, out=None)


def prepare(case, seed):
    dev = _dev()
    with torch.no_grad():
        if case["kind"].startswith("llama"):
            return _prepare_llama(case, seed, dev)
        if case["kind"].startswith("hybrid"):
            return _prepare_hybrid(case, seed, dev)
        return _prepare_moe(case, seed, dev)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return dict(logits=state["logits"], state=state["out"])
    with torch.no_grad():
        got = state["call"]()
    return got if state["out"] is None else dict(logits=got, state=state["out"])


# ---- what a pass cannot do without -----------------------------------------------------------------------------------


def work(case):
    if case["kind"] == "moe":
        d, ne, ni, top, ff = _moe_sizes(case)
        mats, t = (3 if case["form"] == "glu" else 2), case["tokens"]
        real = t * top * ne / (ne + ni)
        used = ne * (1.0 - (1.0 - 1.0 / ne) ** real)
        return dict(bytes=used * mats * d * ff * 2 + (ne + ni) * d * 2 + t * d * 4 + t * top * 8,
                    flops=2.0 * real * mats * d * ff + 2.0 * t * d * (ne + ni))
    lens = _lens(case)
    decode = "decode" in case["kind"] or case["kind"] == "llama_long"
    T = len(lens) if decode else sum(lens)
    seen = [n + 1 for n in lens] if decode else [(n + 1) / 2 for n in lens]   # keys per query, on average
    pairs = sum(seen) if decode else sum(n * s for n, s in zip(lens, seen))
    B = len(lens)
    if case["kind"].startswith("llama"):
        c = _llama_config(case)
        d, f, V, H, G, D = c.hidden_size, c.intermediate_size, c.vocab_size, c.num_heads, c.num_kv_heads, c.head_dim
        per = d * (H + 2 * G) * D + H * D * d + 3 * d * f
        eb = 1 if case["kind"] == "llama_long" else 2
        kv = 2 * G * D * eb
        keys = sum(seen) if decode else 0
        return dict(bytes=LAYERS * (2 * per + keys * kv + T * kv) + V * d * 2 + T * d * 2 + B * V * 2,
                    flops=LAYERS * (2.0 * T * per + 4.0 * pairs * H * D) + 2.0 * B * V * d)
    cfg = _hybrid_config(case)
    d, V = cfg.hidden_size, cfg.vocab_size
    shapes = DESIGNS[case["design"]][0].tensor_shapes(cfg)
    mats = sum(math.prod(s) for n, s in shapes.items() if n.startswith("l") and len(s) == 2)
    nbytes, flops = 2.0 * mats + V * d * 2 + T * d * 2 + B * V * 4, 2.0 * T * mats + 2.0 * B * V * d

    def mixer(m):
        nonlocal nbytes, flops
        if m.kind == "parallel":
            mixer(m.left)
            mixer(m.right)
        elif m.kind in ("mlstm", "delta_rule", "gla", "retention"):
            st = m.heads * m.dim * m.vdim
            nbytes += B * st * 4 * (2 if decode else 1)
            flops += T * st * (6.0 if m.kind == "delta_rule" else 4.0)
        elif m.kind == "latent_attention":
            nbytes += (sum(seen) if decode else T) * (m.kv_rank + m.rot_dim) * 2
            # keys and values materialised per head (the cheaper form for a prompt), or one latent row for all (a decode step)
            flops += 2.0 * pairs * m.heads * ((2 * m.kv_rank + m.rot_dim) if decode else (m.dim + m.rot_dim + m.vdim))
        else:
            w = m.window or (1 << 30)
            if decode:
                n = [min(s, w + m.keep_first) for s in seen]
                vis = sum(n)
                nbytes += vis * m.kv_heads * (m.dim + m.vdim) * 2
            else:
                vis = sum(n * (n + 1) / 2 - (max(0, n - w) * (max(0, n - w) + 1) / 2) for n in lens)
                if m.pool and m.window:
                    vis += sum(max(0, n - w) ** 2 / 2 / m.pool for n in lens)
                nbytes += T * m.kv_heads * (m.dim + m.vdim) * 2
            flops += 2.0 * vis * m.heads * (m.dim + m.vdim)

    for l in cfg.layers:
        mixer(l.mixer)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # bfloat16 activations between the products: measured against exact(), about four times that
    if case["kind"] == "moe":
        return {"rel": 0.012, "max": 0.1, "differ": 1e-4}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits, from the models' equations -------------------------------------------------------------------


def _d(t):
    return t.to(F64)


def _rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _mm(x, w):
    return x @ _d(w).t()


def _table(rot, dims, dev):
    """cos and sin [8192 .., dims / 2] of a rotation's positions, as functions of a position tensor."""
    base = float(rot["base"])
    inv = base ** (-torch.arange(0, dims, 2, dtype=F64, device=dev) / dims)
    sc, mag = rot.get("scaling"), 1.0
    if sc and "low" in sc:
        wl = 2 * math.pi / inv
        s = ((sc["original"] / wl - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        mid = (1 - s) * inv / sc["factor"] + s * inv
        inv = torch.where(wl < sc["original"] / sc["high"], inv, torch.where(wl > sc["original"] / sc["low"], inv / sc["factor"], mid))
    elif sc and "fast" in sc:
        at = lambda t: dims * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
        r = ((torch.arange(dims // 2, dtype=F64, device=dev) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        inv = inv / sc["factor"] * r + inv * (1 - r)
        mag = 0.1 * math.log(sc["factor"]) + 1.0
    elif sc:
        inv = inv / sc["factor"]
    return lambda pos: ((_d(pos)[:, None] * inv).cos() * mag, (_d(pos)[:, None] * inv).sin() * mag)


def _rot(x, cs, dims, back=False):
    """x [T, heads, n]: entry i of the first dims turns with entry i + dims / 2."""
    c, s = cs[0][:, None], (-cs[1] if back else cs[1])[:, None]
    h = dims // 2
    u, v = x[..., :h], x[..., h:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


class _Seqs:
    """The step's token ranges in 64-bit arithmetic: lens[b] cached tokens before the range (decode: one token each)."""

    def __init__(self, case, dev):
        lens = _lens(case)
        self.decode = not case["kind"].endswith("prefill")
        self.n = [1] * len(lens) if self.decode else lens
        self.past = lens if self.decode else [0] * len(lens)
        at = [0]
        for n in self.n:
            at.append(at[-1] + n)
        self.range = list(zip(at, at[1:]))
        self.pos = torch.cat([torch.arange(p, p + n, device=dev) for p, n in zip(self.past, self.n)])
        self.pages = _pages([p + n for p, n in zip(self.past, self.n)])[0]
        # for the recurrences: token t of every sequence at once, longest sequences first
        self.order = sorted(range(len(lens)), key=lambda b: -self.n[b])
        self.steps = []
        for t in range(max(self.n)):
            live = [b for b in self.order if self.n[b] > t]
            self.steps.append(torch.tensor([self.range[b][0] + t for b in live], device=dev))

    def cached(self, pages, b):
        """The rows that sequence b had in a paged cache [NB, BS, ...] before the step."""
        idx = torch.tensor(self.pages[b], device=pages.device)
        return _d(pages[idx].flatten(0, 1)[:self.past[b]])


def _attend(q, k, v, pos, scale, hidden, sink=None):
    """q [n, H, D], k [m, H, D], v [m, H, Dv]; hidden [n, m]: pairs that are not seen.  Returns [n, H, Dv]."""
    s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) * scale
    s = s.masked_fill(hidden[None], float("-inf"))
    if sink is not None:
        s = torch.cat([s, sink[:, None, None].expand(-1, s.shape[1], 1)], -1)
    a = torch.softmax(s, -1)[..., :k.shape[0]]
    return torch.matmul(a, v.transpose(0, 1).contiguous()).transpose(0, 1)


def _scan(seqs, S, step, T, H, Dv):
    """Runs step(S[live], token rows) -> read-out over the sequences side by side; S [B, H, D, Dv] in batch order."""
    order = torch.tensor(seqs.order, device=S.device)
    Sx = S[order].clone()
    out = torch.empty(T, H, Dv, dtype=F64, device=S.device)
    for rows in seqs.steps:
        n = rows.numel()
        out[rows] = step(Sx, n, rows)
    S = S.clone()
    S[order] = Sx
    return out, S


def _read(S, q):
    return torch.matmul(q.unsqueeze(-2), S).squeeze(-2)


class _Hybrid:
    """Forward of the designs' mechanisms, whole sequences at a time, float64."""

    def __init__(self, case, seed, dev):
        self.c, mod = _hybrid_dict(case), DESIGNS[case["design"]][0]
        cfg = _hybrid_config(case)
        self.W = _hybrid_tensors(cfg, mod, dev, seed)
        self.dev, self.seqs, self.eps = dev, _Seqs(case, dev), float(self.c["norm"]["eps"])
        self.T = self.seqs.range[-1][1]
        self.B = len(self.seqs.n)
        self.v_first, self.S, self.state = None, {}, None

    def before(self, name, li, shape):
        """A recurrent state before the step."""
        if self.state is None:
            return torch.zeros(self.B, *shape, dtype=F64, device=self.dev)
        return _d(getattr(self.state, name)[li][:self.B])

    def mlstm(self, li, m, h, w):
        H, D, Dv, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        T = self.T
        q, k, v = (_mm(h, w(n)).view(T, H, -1) for n in "qkv")
        q = q * D ** -0.5
        soft = lambda z: cap * torch.tanh(z / cap)  # noqa: E731
        ig = soft(_mm(h, w("i")) + _d(w("i.b")))
        fg = torch.nn.functional.logsigmoid(soft(_mm(h, w("f")) + _d(w("f.b"))))
        order = torch.tensor(self.seqs.order, device=self.dev)
        nn, mm = self.before("n", li, (H, D))[order], self.before("m", li, (H,))[order]

        def step(S, n, r):
            mn = torch.maximum(fg[r] + mm[:n], ig[r])
            a, b = torch.exp(fg[r] + mm[:n] - mn), torch.exp(ig[r] - mn)
            S[:n] = a[..., None, None] * S[:n] + (b[..., None] * k[r]).unsqueeze(-1) * v[r].unsqueeze(-2)
            nn[:n] = a[..., None] * nn[:n] + b[..., None] * k[r]
            mm[:n] = mn
            den = torch.maximum((nn[:n] * q[r]).sum(-1).abs(), torch.exp(-mn)) + 1e-6
            return _read(S[:n], q[r]) / den[..., None]

        o, self.S[li] = _scan(self.seqs, self.before("S", li, (H, D, Dv)), step, T, H, Dv)
        y = _rms(o, self.eps).reshape(T, -1) * _d(w("norm")) * torch.sigmoid(_mm(h, w("g")))
        return _mm(y, w("o"))

    def latent(self, li, m, h, w):
        H, D, R, Dv, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        tab, dims = _table(m["rot"], m["rot"]["dims"], self.dev), m["rot"]["dims"]
        cs = tab(self.seqs.pos)
        q = _mm(h, w("q")).view(self.T, H, D + R)
        q = torch.cat([q[..., :D], _rot(q[..., D:], cs, dims)], -1)
        kv = _mm(h, w("dkv"))
        row = torch.cat([_rms(kv[:, :rank], self.eps) * _d(w("dkv.norm")), _rot(kv[:, None, rank:], cs, dims)[:, 0]], -1)
        out = torch.empty(self.T, H, Dv, dtype=F64, device=self.dev)
        for b, (t0, t1) in enumerate(self.seqs.range):
            x = row[t0:t1] if not self.seqs.decode else torch.cat([self.seqs.cached(self.state.lat[li], b), row[t0:t1]])
            k = torch.cat([_mm(x[:, :rank], w("uk")).view(-1, H, D), x[:, None, rank:].expand(-1, H, -1)], -1)
            v = _mm(x[:, :rank], w("uv")).view(-1, H, Dv)
            p = self.seqs.pos[t0:t1]
            hid = torch.arange(x.shape[0], device=self.dev)[None] > p[:, None]
            out[t0:t1] = _attend(q[t0:t1], k, v, p, m["scale"], hid)
        out = out * torch.sigmoid(_mm(h, w("g")))[..., None]
        return _mm(out.reshape(self.T, -1), w("o"))

    def attention(self, li, m, h, w, form):
        """form "window" (normed, rotated, sinks, kept first tokens, mixed values), "pooled" (values are the unrotated keys,
        block means before the window) or "sink" (causal, rotated values turned back, a gate per column)."""
        H, G, D, Dv, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.T
        rot, mask = m["rot"], m.get("mask") or {}
        dims, cs = rot["dims"], _table(rot, rot["dims"], self.dev)(self.seqs.pos)
        q, k = _mm(h, w("q")).view(T, H, D), _mm(h, w("k")).view(T, G, D)
        v = k if form == "pooled" else _mm(h, w("v")).view(T, G, Dv)
        if form != "pooled":
            q, k = _rms(q, self.eps) * _d(w("q.norm")), _rms(k, self.eps) * _d(w("k.norm"))
        q, k = _rot(q, cs, dims), _rot(k, cs, dims)
        if form == "window":
            if self.v_first is None:
                self.v_first = v
            else:
                lam = _d(w("vmix"))
                v = (1 - lam) * v + lam * self.v_first
        if form == "sink":
            cv = _table(dict(base=rot["base"]), Dv, self.dev)(self.seqs.pos)
            v = _rot(v, cv, Dv)
        size, keep, pool = mask.get("size", 0), mask.get("keep_first", 0), mask.get("pool", 0)
        sink = None if form == "pooled" else _d(w("sink"))
        rep = lambda x: x.repeat_interleave(H // G, 1)  # noqa: E731
        out = torch.empty(T, H, Dv, dtype=F64, device=self.dev)
        for b, (t0, t1) in enumerate(self.seqs.range):
            kk, vv, p = k[t0:t1], v[t0:t1], self.seqs.pos[t0:t1]
            if self.seqs.decode:
                kk = torch.cat([self.seqs.cached(self.state.kc[li], b), kk])
                vv = torch.cat([self.seqs.cached(self.state.vc[li], b), vv])
            j = torch.arange(kk.shape[0], device=self.dev)[None]
            hid = j > p[:, None]
            if size:
                hid = hid | ((p[:, None] - j >= size) & (j >= keep))
            nb = max(0, (int(p.max()) - size + 1) // pool) if pool else 0
            if nb:
                mean = lambda x: x[:nb * pool].view(nb, pool, G, -1).mean(1)  # noqa: E731
                e = torch.arange(nb, device=self.dev)[None]
                hid = torch.cat([hid, (e + 1) * pool - 1 + size > p[:, None]], 1)
                kk, vv = torch.cat([kk, mean(kk)]), torch.cat([vv, mean(vv)])
            out[t0:t1] = _attend(q[t0:t1], rep(kk), rep(vv), p, m["scale"], hid, sink)
        if form == "sink":
            out = _rot(out, cv, Dv, back=True)
        out = out.reshape(T, -1)
        if form == "window":
            out = (out.view(T, H, Dv) * torch.sigmoid(_mm(h, w("g")))[..., None]).reshape(T, -1)
        elif form == "sink":
            out = out * torch.sigmoid(_mm(h, w("g")))
        return _mm(out, w("o"))

    def gated_read(self, h, o, w, norm):
        g = _mm(h, w("g"))
        return _mm((_rms(o, self.eps) * norm).reshape(self.T, -1) * g * torch.sigmoid(g), w("o"))

    def delta(self, li, m, h, w):
        HK, H, D, Dv, K, T = m["kv_heads"], m["heads"], m["dim"], m["vdim"], m["conv"], self.T
        x = torch.cat([_mm(h, w(n)) for n in "qkv"], -1)
        taps = torch.cat([_d(w(n + ".conv")) for n in "qkv"], 0)
        y = torch.empty_like(x)
        past = self.before("hist", li, (K - 1, x.shape[1]))
        for b, (t0, t1) in enumerate(self.seqs.range):
            ext = torch.cat([past[b], x[t0:t1]])
            acc = sum(ext[i:i + t1 - t0] * taps[:, i] for i in range(K))
            y[t0:t1] = acc * torch.sigmoid(acc)
        q, k = y[:, :HK * D].view(T, HK, D), y[:, HK * D:2 * HK * D].view(T, HK, D)
        unit = lambda z: z * torch.rsqrt(z.pow(2).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k = (z.repeat_interleave(H // HK, 1) for z in (unit(q) * D ** -0.5, unit(k)))
        v = y[:, 2 * HK * D:].view(T, H, Dv)
        dec = torch.exp(-torch.exp(_d(w("A_log"))) * torch.nn.functional.softplus(_mm(h, w("a")) + _d(w("dt_bias"))))
        beta = torch.sigmoid(_mm(h, w("b")))

        def step(S, n, r):
            s = S[:n] * dec[r][..., None, None]
            u = beta[r][..., None] * (v[r] - _read(s, k[r]))
            S[:n] = s + k[r].unsqueeze(-1) * u.unsqueeze(-2)
            return _read(S[:n], q[r])

        o, self.S[li] = _scan(self.seqs, self.before("S", li, (H, D, Dv)), step, T, H, Dv)
        return self.gated_read(h, o, w, _d(w("norm")))

    def gla(self, li, m, h, w):
        H, D, Dv, T = m["heads"], m["dim"], m["vdim"], self.T
        q, k, v = (_mm(h, w(n)).view(T, H, -1) for n in "qkv")
        z = _mm(_mm(h, w("a1")), w("a2")) + _d(w("a2.b"))
        dec = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, H, D)

        def step(S, n, r):
            S[:n] = S[:n] * dec[r].unsqueeze(-1) + k[r].unsqueeze(-1) * v[r].unsqueeze(-2)
            return _read(S[:n], q[r] * D ** -0.5)

        o, self.S[li] = _scan(self.seqs, self.before("S", li, (H, D, Dv)), step, T, H, Dv)
        return self.gated_read(h, o, w, _d(w("norm")))

    def retention(self, li, m, h, w):
        H, D, Dv, T = m["heads"], m["dim"], m["vdim"], self.T
        cs, dims = _table(m["rot"], m["rot"]["dims"], self.dev)(self.seqs.pos), m["rot"]["dims"]
        q, k, v = (_mm(h, w(n)).view(T, H, -1) for n in "qkv")
        q, k = _rot(q, cs, dims), _rot(k, cs, dims) * D ** -0.5
        dec = torch.tensor(m["decay"], dtype=F64, device=self.dev)[:, None, None]

        def step(S, n, r):
            S[:n] = S[:n] * dec + k[r].unsqueeze(-1) * v[r].unsqueeze(-2)
            return _read(S[:n], q[r])

        o, self.S[li] = _scan(self.seqs, self.before("S", li, (H, D, Dv)), step, T, H, Dv)
        return self.gated_read(h, o, w, 1.0)

    def mixer(self, i, l, h):
        m, w = l["mixer"], lambda n: self.W[f"l{i}.mix.{n}"]  # noqa: E731
        form = {"zokunex": {"mlstm": self.mlstm, "latent_attention": self.latent},
                "kalesun": {"delta": self.delta, "gla": self.gla, "attention": lambda *a: self.attention(*a, "window")},
                "vogerax": {"attention": lambda *a: self.attention(*a, "pooled")}}[self.c["architecture"].lower()]
        if l["type"] != "parallel":
            return form[l["type"]](i, m, h, w)
        side = lambda s: (lambda n: self.W[f"l{i}.mix.{s}.{n}"])  # noqa: E731
        a = self.attention((i, 0), m["left"], h, side("left"), "sink")
        r = self.retention((i, 1), m["right"], h, side("right"))
        return 0.5 * (_rms(a, self.eps) * _d(w("left.out")) + _rms(r, self.eps) * _d(w("right.out")))

    def forward(self, ids, state=None):
        self.state = state
        kind, eps = self.c["architecture"].lower(), self.eps
        W = lambda n: _d(self.W[n])  # noqa: E731
        x = W("embed")[ids.long()]
        last = torch.tensor([t1 - 1 for _, t1 in self.seqs.range], device=self.dev)
        ln = lambda y: torch.nn.functional.layer_norm(y, y.shape[-1:], eps=eps)  # noqa: E731
        if kind == "vogerax":
            x = x * self.c["embedding"]["scale"]
            ng = self.c["norm"]["groups"]
            gn = lambda y: _rms(y.view(*y.shape[:-1], ng, -1), eps).flatten(-2)  # noqa: E731
        for i, l in enumerate(self.c["layers"]):
            p = f"l{i}."
            for k, name in ((0, "norm1"), (1, "norm2")):
                h = gn(x) * W(p + name) if kind == "vogerax" else x
                if k == 0:
                    y = self.mixer(i, l, h)
                elif kind == "kalesun":
                    g, u = _mm(h, self.W[p + "mlp.gate"]).clamp(max=7.0), _mm(h, self.W[p + "mlp.up"]).clamp(-7.0, 7.0)
                    y = _mm(g * torch.sigmoid(1.702 * g) * (u + 1.0), self.W[p + "mlp.down"])
                else:
                    y = _mm(torch.relu(_mm(h, self.W[p + "mlp.up"])).pow(2), self.W[p + "mlp.down"])
                if kind == "zokunex":
                    x = x + ln(y) * W(p + name)
                elif kind == "kalesun":
                    x = _rms(self.c["postln_alpha"] * x + y, eps) * W(p + name)
                else:
                    x = x + gn(y) * W(p + name + "b")
        x = x[last]
        x = (ln(x) if kind == "zokunex" else gn(x) if kind == "vogerax" else _rms(x, eps)) * W("final.norm")
        return _mm(x, self.W["embed" if kind == "kalesun" else "head"])


def _exact_llama(case, s, dev):
    cfg, w, sb = s["model"].cfg, s["model"].w, s["sb"]
    seqs = _Seqs(case, dev)
    H, G, D, T, eps = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, seqs.range[-1][1], cfg.rms_eps
    cs = _table(dict(base=cfg.rope_theta), D, dev)(seqs.pos)
    x = _d(w.embed[sb.ids.long()])
    num = lambda t: _d(t.view(torch.float8_e4m3fn).to(torch.bfloat16) if t.dtype == torch.uint8 else t)  # noqa: E731
    for l, lw in enumerate(w.layers):
        qkv = _mm(_rms(x, eps), lw.wqkv)
        q, k, v = qkv[:, :H * D].view(T, H, D), qkv[:, H * D:(H + G) * D].view(T, G, D), qkv[:, (H + G) * D:].view(T, G, D)
        q, k = _rot(q, cs, D), _rot(k, cs, D)
        o = torch.empty_like(q)
        for b, (t0, t1) in enumerate(seqs.range):
            kk, vv, p = k[t0:t1], v[t0:t1], seqs.pos[t0:t1]
            if seqs.decode:
                pg, n = torch.tensor(seqs.pages[b], device=dev), seqs.past[b]
                kk = torch.cat([num(s["kv"].k[l][pg]).permute(0, 2, 1, 3).flatten(0, 1)[:n], kk])
                vv = torch.cat([num(s["kv"].v[l][pg]).permute(0, 3, 1, 2).flatten(0, 1)[:n], vv])
            hid = torch.arange(kk.shape[0], device=dev)[None] > p[:, None]
            qq = q[t0:t1].view(t1 - t0, G, H // G, D)
            sc = torch.matmul(qq.permute(1, 2, 0, 3).reshape(G, -1, D), kk.permute(1, 2, 0).contiguous()) * D ** -0.5
            a = torch.softmax(sc.view(G, H // G, t1 - t0, -1).masked_fill(hid, float("-inf")), -1)
            ob = torch.matmul(a.view(G, -1, a.shape[-1]), vv.transpose(0, 1).contiguous()).view(G, H // G, t1 - t0, D)
            o[t0:t1] = ob.permute(2, 0, 1, 3).reshape(t1 - t0, H, D)
        x = x + _mm(o.reshape(T, -1), lw.wo)
        gu = _mm(_rms(x, eps), lw.w_gu)
        f = gu.shape[1] // 2
        x = x + _mm(torch.nn.functional.silu(gu[:, :f]) * gu[:, f:], lw.w_down)
    last = torch.tensor([t1 - 1 for _, t1 in seqs.range], device=dev)
    return _mm(_rms(x[last], eps), w.lm_head)


def _exact_moe(case, seed, dev):
    t = _moe_inputs(case, seed, dev)
    _, ne, _, top, ff = _moe_sizes(case)
    h = _d(t["h"])
    z = _mm(h, t["w_r"])
    if case["form"] == "glu":
        val, idx = torch.topk(z + _d(t["b"]), top, dim=-1)
        wt = torch.softmax(val, -1)
    else:
        s = torch.softmax(z, -1)
        idx = torch.topk(s + _d(t["b"]), top, dim=-1).indices
        wt = torch.gather(s, 1, idx)
    y = ((idx >= ne) * wt).sum(-1, keepdim=True) * h
    for e in range(ne):
        tok, kk = torch.nonzero(idx == e, as_tuple=True)
        if tok.numel():
            u = _mm(h[tok], t["w_up"][e])
            if case["form"] == "glu":
                g, u = u[:, :ff].clamp(max=7.0), u[:, ff:].clamp(-7.0, 7.0)
                u = g * torch.sigmoid(1.702 * g) * (u + 1.0)
            else:
                u = torch.nn.functional.gelu(u)
            y.index_add_(0, tok, _mm(u, t["w_down"][e]) * wt[tok, kk][:, None])
    return dict(idx=None, wt=wt, y=y)


def exact(case, seed):
    dev = _dev()
    with torch.no_grad():
        if case["kind"] == "moe":
            return _exact_moe(case, seed, dev)
        s = _prepare_llama(case, seed, dev) if case["kind"].startswith("llama") else _prepare_hybrid(case, seed, dev)
        none = [None] * len(s["out"])
        if case["kind"].startswith("llama"):
            return dict(logits=_exact_llama(case, s, dev), state=none)
        m = _Hybrid(case, seed, dev)
        logits = m.forward(s["sb"].ids, s["kv"] if m.seqs.decode else None)
        for i, (key, t) in enumerate(s["kv"].S.items()):   # the recurrent states come first; the last row is nobody's
            none[i] = torch.cat([m.S[key], _d(t[m.B:])])
        return dict(logits=logits, state=none)
