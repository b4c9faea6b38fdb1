"""The grouped experts (csrc/hybrid/moe_grouped.hip) where their launches change shape: 32-, 128- and 256-row tiles, one and
several workgroups placing the items, weight rows that end inside a 256-row tile, choices that leave experts empty or send every
token to one, single tokens, identity experts and indices that name nobody.  Against the PyTorch reference; the tolerance is
that of the other expert tests (bfloat16 activations between the two products)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def _close(a, b, tol=1.5e-2):
    a, b = a.float(), b.float()
    assert float((a - b).abs().max()) <= tol * (float(b.abs().max()) + 1e-6)


def _choice(kind, g, T, E, top):
    if kind == "skew":   # everybody's first choice is expert 0
        idx = torch.rand(T, E, device=DEV, generator=g)
        idx[:, 0] = 2.0
    else:
        idx = torch.rand(T, E, device=DEV, generator=g)
        if kind == "empty" and E > top:
            idx[:, 1] = -1.0
    idx = idx.topk(top, -1).indices.int()
    wt = torch.rand(T, top, device=DEV, generator=g)
    if kind == "nobody":   # an index that names no expert adds nothing
        idx[::3, -1] = -1
    return idx.contiguous(), wt


@pytest.mark.parametrize("T,d,F,E,top", [(1, 256, 128, 4, 4), (1, 128, 256, 256, 8), (33, 256, 384, 8, 2), (513, 128, 128, 2, 1),
                                         (1100, 256, 256, 4, 4), (3000, 128, 128, 40, 2), (11000, 512, 384, 8, 8),
                                         (9000, 512, 256, 3, 8 // 3)])
@pytest.mark.parametrize("kind", ["even", "skew", "empty", "nobody"])
def test_experts(T, d, F, E, top, kind):
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    g = torch.Generator(device=DEV).manual_seed(T + E)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    h = rnd(T, d).to(BF)
    idx, wt = _choice(kind, g, T, E, top)
    wu, wd = (rnd(E, F, d) * d ** -0.5).to(BF), (rnd(E, d, F) * F ** -0.5).to(BF)
    ident = idx.clone()
    if kind != "nobody":
        ident[::5, 0] = E   # an identity expert
    for act in (0, 1):
        _close(hops.moe_ffn(h, ident, wt, wu, wd, act, BF), ref.moe_ffn(h, ident, wt, wu, wd, act, BF))
    wgu = (rnd(E, 2 * F, d) * d ** -0.5).to(BF)
    tiled = wgu[:, hops.moe_glu_row_order(F).to(DEV)].contiguous()
    _close(hops.moe_glu_ffn(h, idx, wt, tiled, wd, 2.0, 1.702, 1.0, BF, True), ref.moe_glu_ffn(h, idx, wt, wgu, wd, 2.0, 1.702, 1.0, BF))


@pytest.mark.parametrize("T,d,F,E,top", [(768, 2048, 2048, 12, 3), (2051, 2176, 2048, 5, 1), (1300, 1024, 512, 32, 8), (1540, 1024, 512, 32, 8),
                                         (8200, 640, 512, 20, 1)])
@pytest.mark.parametrize("kind", ["even", "skew", "empty", "nobody"])
def test_experts_with_less_than_a_round_of_large_tiles(T, d, F, E, top, kind):
    """From 192 items per expert on, 384 of narrow ones, the 256-row tile takes launches that have fewer tiles than the chip has CUs."""
    test_experts(T, d, F, E, top, kind)


@pytest.mark.parametrize("T", [1, 37, 3000])
def test_no_choice(T):
    """idx [T, 0]: the sum of no experts is zero, whatever the result's memory held."""
    from chronos.ops import hybrid as hops

    d, F, E = 256, 128, 4
    h = torch.randn(T, d, device=DEV).to(BF)
    idx, wt = torch.empty(T, 0, device=DEV, dtype=torch.int32), torch.empty(T, 0, device=DEV)
    wu, wgu, wd = (torch.randn(E, *s, device=DEV).to(BF) for s in ((F, d), (2 * F, d), (d, F)))
    for call in (lambda: hops.moe_ffn(h, idx, wt, wu, wd, 0, BF), lambda: hops.moe_ffn(h, idx, wt, wu, wd, 1, BF),
                 lambda: hops.moe_glu_ffn(h, idx, wt, wgu, wd, 2.0, 1.702, 1.0, BF, True),
                 lambda: hops.moe_glu_ffn(h, idx, wt, wgu, wd, 2.0, 1.702, 1.0, BF)):
        held = torch.full((T, d), float("nan"), device=DEV, dtype=BF)   # the block that the result is likely to get
        del held
        assert torch.equal(call(), torch.zeros_like(h))


def test_experts_in_a_graph():
    """Several replays with new choices in between: the routing is only known on the device."""
    from chronos.ops import hybrid as hops

    g = torch.Generator(device=DEV).manual_seed(3)
    T, d, F, E, top = 2500, 256, 128, 6, 2
    h, wd = torch.randn(T, d, device=DEV, generator=g).to(BF), (torch.randn(E, d, F, device=DEV, generator=g) * 0.1).to(BF)
    tiled = (torch.randn(E, 2 * F, d, device=DEV, generator=g) * 0.06).to(BF)
    idx, wt = _choice("even", g, T, E, top)
    run = lambda: hops.moe_glu_ffn(h, idx, wt, tiled, wd, 7.0, 1.702, 1.0, BF, True)  # noqa: E731
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run()
    for kind in ("even", "skew", "empty", "even"):
        i2, w2 = _choice(kind, g, T, E, top)
        idx.copy_(i2)
        wt.copy_(w2)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, run())
