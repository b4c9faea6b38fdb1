"""Projections of many rows that no measured plan lists (ops/gemm.py many_rows_plan, product_act): what the rule may return, and on
the GPU the routed product and the activations in its epilogue against float64 of the same bfloat16 operands."""
import itertools

import pytest
import torch

from chronos.ops import gemm as G

DEV = "cuda"


def test_rule_returns_what_the_kernels_take():
    for m, n, k in itertools.product((128, 129, 1000, 8192, 100000), (4, 6, 60, 512, 5632, 20224), (32, 64, 96, 1024, 4096, 1 << 20)):
        plan = G.many_rows_plan(m, n, k)
        if plan is not None:
            assert plan[0] in (19, 32, 88) and G._pp_valid(plan[0], n, k, G.PP_PLAIN, 1, m)
            assert (max(m, n) + 256) * k * 2 < 1 << 31
            assert k // 64 % plan[1] == 0 and (plan[1] == 1 or (plan[0] == 88 and G._pp_valid(88, n, k, G.PP_PLAIN, plan[1], m)
                                                                and -(-m // 256) * -(-n // 256) * plan[1] <= 256))
    assert G.many_rows_plan(8192, 2048, 96) is None and G.many_rows_plan(8192, 2050, 128) is None
    assert G.many_rows_plan(128, 64, 4096) is None         # too few tiles without a split of K
    assert G.many_rows_plan(1000, 4096, 11008)[1] > 1      # ... with one
    assert G.many_rows_plan(2446, 1536, 1024) == G.many_rows_plan(2550, 1536, 1024)   # rows count in 128s
    assert G.many_rows_plan(4096, 6144, 4096) is None      # the measured plan's own


def test_measured_plan_and_modes_come_first(monkeypatch):
    assert G.many_rows_plan(8192, 2048, 2048) is not None
    for mode in ("lib", "own"):
        monkeypatch.setattr(G, "PP_MODE", mode)
        assert G.many_rows_plan(8192, 2048, 2048) is None


def test_registered_kernels_get_their_products(monkeypatch):
    """A product that a kernel is registered for is linear()'s: no launch that takes it along with a sum, rows behind or an activation."""
    import chronos.ops as ops

    calls = []

    class Kernels:
        def __getattr__(self, name):
            return lambda *args: calls.append(name) or ("y", "f")

    monkeypatch.setattr(ops, "_k", Kernels)
    x, w = torch.zeros(8, 1024, dtype=torch.bfloat16), torch.zeros(4096, 1024, dtype=torch.bfloat16)
    x2 = torch.zeros(4, 4096, dtype=torch.bfloat16)
    w2 = torch.zeros(4096, 4096, dtype=torch.bfloat16)
    xm = torch.zeros(4096, 1024, dtype=torch.bfloat16)
    monkeypatch.setattr(G, "_custom", [])

    def every():
        return (G.product_slices(x2, w2), G.product_rows(x, w, 4064, 32, None), G.product_act(x, w, 3), G.product_act(xm, w, 5))

    assert None not in every() and calls == ["gemm_slices", "gemm_few", "gemm_few", "gemm_act"]
    G.register(lambda m, n, k: (m, n, k) in ((4, 4096, 4096), (8, 4064, 1024), (8, 4096, 1024), (4096, 4096, 1024)), lambda x, w: None)
    assert every() == (None, None, None, None) and len(calls) == 4
    G._custom[:] = [(lambda m, n, k: (m, n, k) == (8, 4064, 1025), None)]
    assert None not in every()


# rows behind the product that fill no 4 (the joined matrix ends with them, or has padding), no rows at all, a product off the 4s
@pytest.mark.parametrize("m", [8, 100, 300])
@pytest.mark.parametrize("rows,n0,nf,one", [(1030, 1024, 6, None), (1029, 1024, 5, None), (1056, 1024, 6, True), (1032, 1024, 6, True), (1056, 1024, 0, None),
                                            (1024, 1002, 22, None)])
def test_rows_behind_that_one_launch_does_not_take(monkeypatch, m, rows, n0, nf, one):
    """... stay with two: what gemm_ring and gemm_few refuse (n0 in 4s, n0 + nf rows in 4s, rows behind there) does not reach them."""
    import chronos.ops as ops

    class Kernels:
        def gemm_ring(self, x, w, cfg, split, mode, n0, nf, *more):
            assert n0 % 4 == 0 and nf > 0 and (n0 + nf + 3) // 4 * 4 <= w.shape[0]
            return "y", "f"

        def gemm_few(self, x, w, cfg, mode, n0, nf, *more):
            assert n0 % 4 == 0 and nf > 0 and n0 + nf <= w.shape[0] and w.shape[0] % 32 == 0
            return "y", "f"

    monkeypatch.setattr(ops, "_k", Kernels)
    x, w = torch.zeros(m, 1024, dtype=torch.bfloat16), torch.zeros(rows, 1024, dtype=torch.bfloat16)
    got = G.product_rows(x, w, n0, nf, None)
    assert got is None if one is None or (m <= 64 and rows % 32) else got == ("y", "f")
    h = torch.zeros(1, 1024, dtype=torch.bfloat16)
    assert n0 % 4 == 0 or G.join_config(h, w, 0, n0) == 0


def _operands(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    return torch.randn(m, k, device=DEV, generator=g).bfloat16(), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).bfloat16()


def _check(y, want):
    """float32 sums (2^-24 sqrt(K) of the root mean square) and one rounding to bfloat16: 2^-8 |y| + 1e-4 rms(y)."""
    assert y.dtype == torch.bfloat16 and y.shape == want.shape
    assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + 1e-4 * want.square().mean().sqrt()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(128, 4096, 64), (129, 4100, 192), (2446, 1536, 1024), (2446, 5632, 1024), (1000, 8196, 64), (8192, 260, 512),
                                   (1000, 4096, 11008), (600, 4096, 14336), (300, 2048, 8192)])
def test_linear(m, n, k):
    from chronos import ops

    x, w = _operands(m, n, k)
    assert G.many_rows_plan(m, n, k) is not None
    _check(ops.linear(x, w), x.double() @ w.double().t())
    y3 = ops.linear(x.view(1, m, k), w)
    assert y3.shape == (1, m, n) and torch.equal(y3[0], ops.linear(x, w))


@pytest.mark.gpu
def test_other_forms_keep_their_way():
    """Column ranges, transposed weights, addresses off 16 bytes and products that gradients have to see."""
    from chronos import ops

    x, w = _operands(512, 4096, 1024)
    want = x[:, :512].double() @ w[:, :512].double().t()
    _check(ops.linear(x[:, :512], w[:, :512]), want)
    _check(ops.linear(x[:, :512].contiguous(), w[:, :512].contiguous().t().contiguous().t()), want)
    flat = torch.empty(512 * 1024 + 1, device=DEV, dtype=torch.bfloat16)
    xo = flat[1:].view(512, 1024).copy_(x)
    _check(ops.linear(xo, w), x.double() @ w.double().t())
    wg = w.clone().requires_grad_(True)
    ops.linear(x, wg).float().sum().backward()
    assert wg.grad is not None


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,unit,other", [(100, 512, 128, False, False), (300, 512, 4096, False, False), (2446, 5632, 1024, True, True),
                                              (4100, 8192, 64, True, True), (1000, 768, 320, False, True)])
def test_activations(m, n, k, unit, other):
    """Either way of the rule: in the product's epilogue (unit: the gated unit's, other: the others'), or a pass of its own on the rounded
    product.  The epilogue's elements one by one: test_gemm_slab_gpu.py."""
    from chronos.ops import hybrid as H

    x, w = _operands(m, n, k)
    assert (G.product_act(x, w, 3) is not None) == unit
    assert (G.product_act(x, w, 4) is not None) == other and (G.product_act(x, w, 5) is not None) == other
    h = x.double() @ w.double().t()
    F = n // 2
    for limit, slope, shift in ((float("inf"), 1.0, 0.0), (0.75, 1.702, 1.0)):
        g, u = h[:, :F].clamp(max=limit), h[:, F:].clamp(-limit, limit)
        want = g * torch.sigmoid(slope * g) * (u + shift)
        y = H.matmul_glu(x, w, limit, slope, shift, torch.bfloat16)
        assert ((y.double() - want).norm() / want.norm()).item() < 2 ** -7   # three roundings to bfloat16 at most
    for kind, want in ((H.ACT_RELU2, h.relu() ** 2), (H.ACT_GELU, torch.nn.functional.gelu(h))):
        y = H.matmul_act(x, w, kind)
        assert ((y.double() - want).norm() / want.norm()).item() < 2 ** -7
