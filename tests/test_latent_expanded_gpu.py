"""Latent attention of whole prompts with keys and values written out (csrc/hybrid/latent_expanded.hip): the kernel against
float64 attention of the same operands, and a model's prompt step against its own step through the cached latents.

Tolerance: the softmax weights and the result are rounded to bfloat16, at most 2^-8 of each: the sum over keys errs by at most 2^-8 of
the sum of |weight value| (random values: less than 2^-8 of the result's norm, the roundings being independent), and the result's own
rounding adds as much; float32 sums and exponentials add 1e-5.  Checked: norm of the difference below 2^-8 of the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,D,R,Dv", [(3, 128, 64, 128), (2, 64, 32, 64), (2, 40, 24, 48), (1, 120, 0, 16), (2, 8, 8, 128)])
@pytest.mark.parametrize("lens,extra", [([1, 33, 0, 300, 128, 257, 64], ""), ([31, 32, 65], "sink"), ([200, 17], "window"),
                                        ([130, 129], "gate"), ([3, 1], "cols"), ([700] * 90, "many")])
def test_kernel(H, D, R, Dv, lens, extra):
    from chronos.ops import hybrid as hops

    T, window = sum(lens), 37 if extra == "window" else 0
    g = torch.Generator(device=DEV).manual_seed(H * D + Dv + T)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    wide = rnd(T, H * (D + R) + 8).bfloat16()
    q = wide[:, :H * (D + R)].view(T, H, D + R)
    kv, kr = rnd(T, H, D + Dv).bfloat16(), rnd(T, R + 8).bfloat16()[:, :R]
    sink = rnd(H) if extra == "sink" else None
    gate = rnd(T, H) if extra == "gate" else None
    cols = rnd(T, H * Dv + 5).bfloat16() if extra == "cols" else None
    qs = [0]
    for n in lens:
        qs.append(qs[-1] + n)
    store = torch.full((T, H * Dv + 4), 7.0, device=DEV).bfloat16()
    scale = (D + R) ** -0.5
    o = hops.latent_expanded(q, kv, kr, torch.tensor(qs, dtype=torch.int32, device=DEV), gate, cols, 5, sink, scale, max(lens), window,
                             store[:, :H * Dv].view(T, H, Dv))
    assert torch.equal(store[:, H * Dv:], torch.full_like(store[:, H * Dv:], 7.0))
    for b, n in enumerate(lens if extra != "many" else lens[:2]):
        if n == 0:
            continue
        sl = slice(qs[b], qs[b + 1])
        k = torch.cat([kv[sl, :, :D], kr[sl, None].expand(n, H, R)], -1).double()
        s = torch.matmul(q[sl].double().transpose(0, 1), k.permute(1, 2, 0)) * scale
        i = torch.arange(n, device=DEV)
        hide = i[None] > i[:, None]
        if window:
            hide |= i[None] <= i[:, None] - window
        s.masked_fill_(hide, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.double().view(H, 1, 1).expand(H, n, 1)], -1)
        want = torch.matmul(torch.softmax(s, -1)[..., :n], kv[sl, :, D:].double().transpose(0, 1)).transpose(0, 1)
        if gate is not None:
            want = want * torch.sigmoid(gate[sl].double())[..., None]
        if cols is not None:
            want = want * torch.sigmoid(cols[sl, 5:].double()).view(n, H, Dv)
        assert float((o[sl].double() - want).norm() / want.norm()) < 2 ** -8, (b, n)


def test_longest_beyond_the_tokens():
    """``max_q`` sizes the launch: more than there are tokens is no error."""
    from chronos.ops import hybrid as hops

    q, kv, kr = torch.randn(40, 2, 96, device=DEV).bfloat16(), torch.randn(40, 2, 128, device=DEV).bfloat16(), torch.randn(40, 32, device=DEV).bfloat16()
    qs = torch.tensor([0, 33, 40], dtype=torch.int32, device=DEV)
    a, b = (hops.latent_expanded(q, kv, kr, qs, None, None, -1, None, 0.1, most) for most in (33, 1 << 20))
    assert torch.equal(a, b)


@pytest.mark.parametrize("rank", [256, 64])
def test_prompt_step(rank):
    """The same latents in the first layer's cache, logits within the two forms' rounding (of different intermediates to bfloat16, 2^-9 each
    and some ten of them, in 2 of 4 layers: 2^-9 sqrt(20) = 0.009, taken three times); a batch whose positions were touched, or whose sequences continue, takes the cached latents."""
    from chronos.models import zokunex
    from chronos.models.hybrid import HybridDecoder
    from chronos.ops import hybrid as hops
    from chronos.utils import design_bench as db

    c = db.zokunex_config(dict(db.SIZES["1k"], a=(8, 64, 32, 64, rank)))
    for layer in c["layers"]:   # dense layers: a router's choice between near-equal experts is no rounding
        layer["mlp"] = c["layers"][0]["mlp"]
    cfg = zokunex.config_from_dict(c, name="z", max_position=1024)
    m = HybridDecoder(cfg, zokunex.pack_weights(cfg, zokunex.random_tensors(cfg, 0), torch.device(DEV), torch.bfloat16),
                      torch.device(DEV), 1024, torch.bfloat16)
    g = torch.Generator().manual_seed(5)
    lens = [600, 1, 77]
    ids = [torch.randint(0, cfg.vocab_size, (n,), generator=g).tolist() for n in lens]
    bts, at = [], 1
    for n in lens:
        bts.append(list(range(at, at + 38)))
        at += 38
    calls = []
    real = hops.latent_expanded

    def counted(*a, **k):
        calls.append(1)
        return real(*a, **k)

    hops.latent_expanded = counted
    try:
        out = []
        for fresh in (True, False, None):
            cache = m.make_cache(at, 16, 3)
            sb = m.prefill_batch(ids, [0, 0, 0], bts, [0, 1, 2])
            assert sb.fresh is not None
            if fresh is False:
                sb.fresh = None
            elif fresh is None:
                sb.pos.add_(0)
            before = len(calls)
            out.append((m.forward(sb, cache).double(), [t.clone() for t in cache.lat.values()]))
            assert (len(calls) > before) == (fresh is True)
        assert m.prefill_batch(ids, [0, 16, 0], bts, [0, 1, 2]).fresh is None
        before = len(calls)   # few tokens: the form with fewer launches
        m.forward(m.prefill_batch([ids[2]], [0], bts[2:], [2]), cache)
        assert len(calls) == before
    finally:
        hops.latent_expanded = real
    assert torch.equal(out[1][0], out[2][0])
    assert torch.equal(out[0][1][0], out[1][1][0])
    assert float((out[0][0] - out[1][0]).norm() / out[1][0].norm()) < 0.03


def test_captured_step(monkeypatch):
    """A prompt step captured while its sequences start at position 0 and replayed after its positions have moved on: the graph must read
    the cached latents, as the same step run eagerly does."""
    from chronos.models import hybrid, zokunex
    from chronos.utils import design_bench as db

    monkeypatch.setattr(hybrid, "EXPAND_MIN", 0)
    c = db.zokunex_config(dict(db.SIZES["1k"], a=(8, 64, 32, 64, 128)))
    for layer in c["layers"]:
        layer["mlp"] = c["layers"][0]["mlp"]
    cfg = zokunex.config_from_dict(c, name="z", max_position=1024)
    m = hybrid.HybridDecoder(cfg, zokunex.pack_weights(cfg, zokunex.random_tensors(cfg, 0), torch.device(DEV), torch.bfloat16),
                             torch.device(DEV), 1024, torch.bfloat16)
    g = torch.Generator().manual_seed(6)
    tokens = lambda lens: [torch.randint(0, cfg.vocab_size, (n,), generator=g).tolist() for n in lens]  # noqa: E731
    lens, bts = [70, 1, 33], [list(range(1 + 10 * b, 11 + 10 * b)) for b in range(3)]
    step = lambda ids, starts: m.prefill_batch(ids, starts, bts, [0, 1, 2])  # noqa: E731
    ids = tokens(lens)
    with torch.no_grad():
        cache, sb = m.make_cache(31, 16, 3), step(ids, [0, 0, 0])
        assert sb.fresh is not None
        m.forward(sb, cache)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m.forward(sb, cache)
        for starts in ([32, 16, 48], [0, 0, 0], [16, 80, 1]):
            prefix, own = tokens(starts), m.make_cache(31, 16, 3)
            some = [b for b in range(3) if starts[b]]
            for to in (cache, own):
                if some:
                    m.forward(m.prefill_batch([prefix[b] for b in some], [0] * len(some), [bts[b] for b in some], some), to)
            now = step(ids, starts)
            want = m.forward(now, own)
            for name in ("pos", "ctx_len"):
                getattr(sb, name).copy_(getattr(now, name))
            graph.replay()
            torch.cuda.synchronize()
            if some:
                assert torch.equal(y, want), starts
            else:   # (run eagerly it takes the other form; tolerance as above)
                assert float((y - want).norm() / want.norm()) < 0.03
