"""Launches that took over a neighbour's work: few-row products with float32 rows or an activation behind (gemm_few), the low-rank decays in
one kernel, the embedding's two copies, the convolution that rewrites its history, the plain layer norm of float rows."""
import pytest
import torch

DEV = "cuda"
BF = torch.bfloat16
pytestmark = pytest.mark.gpu


def _g(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _check(y, want):
    """float32 sums and one rounding to bfloat16: 2^-8 |y| + 1e-4 rms(y)."""
    assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + 1e-4 * want.square().mean().sqrt()).all()


@pytest.mark.parametrize("m", [1, 2, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n0,nf,k", [(512, 8, 64), (1040, 13, 576), (3072, 1, 1024), (4, 60, 192)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_rows_behind(m, n0, nf, k, with_bias):
    from chronos.models.hybrid import _stacked
    from chronos.ops import gemm as G, hybrid as H

    g = _g(m + n0 + nf)
    x, a, b = (torch.randn(s, device=DEV, generator=g).to(BF) for s in ((m, k), (n0, k), (nf, k)))
    bias = torch.randn(nf, device=DEV, generator=g) if with_bias else None
    out = _stacked([a[:n0 // 2], a[n0 // 2:]], b, lambda t: t.contiguous(), {}, "a", "b")
    rows, m0, mf = out["joined"]
    assert rows.shape[0] % 32 == 0 and (m0, mf) == (n0, nf) and torch.equal(out["a"], a) and torch.equal(out["b"], b)
    y, yf = G.product_rows(x, *out["joined"], bias)
    _check(y, x.double() @ a.double().t())
    want = x.double() @ b.double().t() + (0 if bias is None else bias.double())
    assert yf.dtype == torch.float32 and yf.shape == (m, nf)
    assert (yf.double() - want).abs().max() <= 2e-6 * k ** 0.5 * want.abs().max()      # float32 sums of exact products
    y2, yf2 = H.matmul_rowdot(x, out["a"], out["b"], bias, out["joined"])
    assert torch.equal(y, y2) and torch.equal(yf, yf2)


_CONFIGS = ((12, (1, 17, 31, 32)), (13, (1, 33, 63, 64)), (14, (1, 15, 16)), (15, (1, 15, 16)), (16, (1, 17, 31, 32)), (17, (1, 33, 63, 64)))


# (gated units take configs of 32 weight rows: a pair of gate and up rows in a workgroup)
@pytest.mark.parametrize("cfg,ms,mode", [(cfg, ms, mode) for cfg, ms in _CONFIGS for mode in (3, 4, 5) if mode > 3 or cfg >= 15])
@pytest.mark.parametrize("n,k", [(32, 64), (96, 192), (2080, 576), (4096, 1024)])
def test_every_activation_of_every_config(cfg, ms, mode, n, k):
    """gemm_few's epilogues element by element.  float32 sums move a value by less than 2e-5 (sums of products of variance 1 / K, activations of
    slope below 3 there, the square's up to 2 |h|), and there is one rounding to bfloat16: 2^-8 |y| + 2e-5 max(1, |h|)."""
    from chronos import ops

    ops.load()
    g = _g(cfg + mode + n + k)
    w = (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)
    F = n // 2
    for m in ms:
        x = torch.randn(m, k, device=DEV, generator=g).to(BF)
        h = x.double() @ w.double().t()
        for limit, slope, shift in ((float("inf"), 1.0, 0.0), (0.75, 1.702, 1.0)) if mode == 3 else ((0.0, 0.0, 0.0),):
            y, rows = torch.ops.chronos.gemm_few(x, w, cfg, mode, 0, 0, None, limit, slope, shift)
            a, u = h[:, :F].clamp(max=limit), h[:, F:].clamp(-limit, limit)
            want = a * torch.sigmoid(slope * a) * (u + shift) if mode == 3 else h.relu() ** 2 if mode == 4 else torch.nn.functional.gelu(h)
            size = torch.maximum(h[:, :F].abs(), h[:, F:].abs()) if mode == 3 else h.abs()
            assert y.dtype == BF and y.shape == want.shape
            assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + 2e-5 * size.clamp(min=1)).all(), (m, limit)


@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(64, 64), (1056, 576), (5632, 1024), (8192, 2048)])
def test_activations(m, n, k):
    from chronos.ops import gemm as G, hybrid as H

    g = _g(m + n + k)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(BF), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)
    h = x.double() @ w.double().t()
    F = n // 2
    # in the product's epilogue, but for gated units of many rows or weights, which stay a launch of their own
    assert G.product_act(x, w, 4) is not None and G.product_act(x, w, 5) is not None
    assert (G.product_act(x, w, 3) is not None) == (m <= 16 or m <= 32 and n * k < 8e6)
    for limit, slope, shift in ((float("inf"), 1.0, 0.0), (0.75, 1.702, 1.0)):
        a, u = h[:, :F].clamp(max=limit), h[:, F:].clamp(-limit, limit)
        want = a * torch.sigmoid(slope * a) * (u + shift)
        y = H.matmul_glu(x, w, limit, slope, shift, BF)
        assert ((y.double() - want).norm() / want.norm()).item() < 2 ** -7
    for kind, want in ((H.ACT_RELU2, h.relu() ** 2), (H.ACT_GELU, torch.nn.functional.gelu(h))):
        y = H.matmul_act(x, w, kind)
        assert ((y.double() - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("T,R,C", [(1, 16, 512), (3, 1, 4), (21, 16, 2048), (700, 16, 4096), (2500, 7, 1028)])
@pytest.mark.parametrize("p", [1.0 / 16, 0.25])
def test_low_rank_decay(T, R, C, p):
    from chronos.ops import hybrid as H

    g = _g(T + R + C)
    a, w, b = (torch.randn(s, device=DEV, generator=g) for s in ((T, R), (R, C), (C,)))
    a[0, 0] = 40.0
    want = torch.sigmoid(b.double() + a.double() @ w.double()) ** p
    ours = H.low_rank_decay(a, w, b, p)
    theirs = H.decay_pow(torch.addmm(b, a, w), p)     # the two launches it replaces
    assert (ours.double() - want).norm() <= 1.05 * (theirs.double() - want).norm() + 1e-7 * want.norm()


@pytest.mark.parametrize("T", [4 * 65535, 4 * 65535 + 1, 300001])
def test_low_rank_decay_of_many_tokens(T):
    """More tokens than a grid's second axis has blocks for."""
    from chronos.ops import hybrid as H

    g = _g(T)
    a, w, b = (torch.randn(s, device=DEV, generator=g) for s in ((T, 2), (2, 4), (4,)))
    want = torch.sigmoid(b.double() + a.double() @ w.double()) ** 0.25
    assert ((H.low_rank_decay(a, w, b, 0.25).double() - want).abs() <= 1e-6).all()   # (values below 1, a few units of the last place)


@pytest.mark.parametrize("d", [64, 1000, 2052])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_embed_both(d, dt):
    from chronos.ops import hybrid as H

    table = torch.randn(50, d, device=DEV, generator=_g(d)).to(dt)
    ids = torch.tensor([3, 49, 0, 3], dtype=torch.int32, device=DEV)
    x, h = H.embed_rows(ids, table, BF, 1.5)
    assert torch.equal(x, table[ids.long()].float() * 1.5) and h.dtype == BF and torch.equal(h, x.to(BF))


@pytest.mark.parametrize("C,K", [(512, 4), (1032, 2), (100, 3), (64, 6)])
def test_one_token_each_convolution(C, K):
    """max_q = 1 gives the bits of the two launches, outputs and history: a first token, one in the middle, a sequence without a token."""
    from chronos.ops import hybrid as H

    g = _g(C + K)
    x, w = torch.randn(3, C, device=DEV, generator=g).to(BF), torch.randn(C, K, device=DEV, generator=g)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    hist = torch.randn(6, K - 1, C, device=DEV, generator=g).to(BF)
    args = (x, w, i32([0, 1, 3]), i32([0, 1, 2, 2, 3]), i32([0, 5, 9, 1]), i32([4, 1, 3, 0]))
    h1, h2 = hist.clone(), hist.clone()
    y1, y2 = H.short_conv(*args, h1, True), H.short_conv(*args, h2, True, max_q=1)
    assert torch.equal(y1, y2) and torch.equal(h1, h2)
    assert torch.equal(h2[3], hist[3]) and torch.equal(h2[4, -1], x[0])


@pytest.mark.parametrize("C,K", [(512, 4), (4104, 3), (8, 2)])
def test_convolution_whatever_max_q_says(C, K):
    """max_q = 1 beside sequences of 0, 1, 2 and 9 tokens: the bits of the two launches, outputs and history."""
    from chronos.ops import hybrid as H

    g = _g(C + K)
    lens = [2, 1, 0, 9, 1]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    q = [sum(lens[:i]) for i in range(len(lens) + 1)]
    x, w = torch.randn(q[-1], C, device=DEV, generator=g).to(BF), torch.randn(C, K, device=DEV, generator=g)
    hist = torch.randn(7, K - 1, C, device=DEV, generator=g).to(BF)
    args = (x, w, i32([b for b, n in enumerate(lens) for _ in range(n)]), i32(q), i32([6, 0, 4, 1, 8]), i32([5, 1, 2, 0, 6]))
    h1, h2 = hist.clone(), hist.clone()
    y1, y2 = H.short_conv(*args, h1, True), H.short_conv(*args, h2, True, max_q=1)
    assert torch.equal(y1, y2) and torch.equal(h1, h2) and torch.equal(h2[2:5], hist[2:5])


@pytest.mark.parametrize("rows,d", [(1, 4), (64, 4096), (7, 1000), (3, 2052), (2, 5000)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_plain_layer_norm(rows, d, dt):
    from chronos.ops import hybrid as H

    x = torch.randn(rows, d, device=DEV, generator=_g(rows + d)) * 3 + 1
    w = torch.randn(d, device=DEV, generator=_g(d))
    want = torch.nn.functional.layer_norm(x.double(), (d,), w.double(), None, 1e-5)
    y = H.layer_norm(x, w, 1e-5, dt)
    assert y.dtype == dt
    tol = 2 ** -8 if dt == BF else 2e-6
    assert ((y.double() - want).abs() <= want.abs() * tol + 2e-6 * want.abs().max()).all()


@pytest.mark.parametrize("m", [2, 16, 31, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(2064, 2048), (4096, 4096), (1040, 14336), (12304, 1024), (4112, 11008)])
def test_large_weights_split(m, n, k):
    """ops.linear where few_rows_plan splits K over workgroups without tickets: twice the same bits, float64 within the roundings."""
    from chronos import ops
    from chronos.ops import gemm as G

    g = _g(m + n + k)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(BF), torch.randn(n, k, device=DEV, generator=g).to(BF)
    want = x.double() @ w.double().t()
    y = ops.linear(x, w)
    _check(y, want)
    assert torch.equal(y, ops.linear(x, w))
    for cfg in (72, 74, 79) if m <= 32 else (38, 39):
        for sk in (2, 4, 8):
            if k // 64 % sk == 0:
                _check(torch.ops.chronos.gemm_split(x, w, cfg, sk), want)


@pytest.mark.parametrize("m", [2, 16, 32])
@pytest.mark.parametrize("n,k", [(4096, 8192), (8192, 4096), (5120, 5120), (8192, 8192)])
def test_library_products_replay(m, n, k):
    """Shapes that few_rows_plan leaves to the library (_library_streams): a captured one gives the eager bits at every replay, with other work between."""
    from chronos import ops
    from chronos.ops import gemm as G

    assert G.few_rows_plan(m, n, k) is None
    g = _g(m + n + k)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(BF), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)
    want = ops.linear(x, w)
    _check(want, x.double() @ w.double().t())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.linear(x, w)
    for _ in range(4):
        y.fill_(float("nan"))
        torch.randn(1 << 20, device=DEV).sum().item()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
