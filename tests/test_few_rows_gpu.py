"""Projections of few rows that no measured plan lists (ops/gemm.py few_rows_plan, the uneven configs of
csrc/kernels/gemm_skinny.hip) against the float64 product of the same bfloat16 operands.

Tolerance: float32 sums of K products, 2^-24 sqrt(K) relative to the root mean square of the result at most (K <= 11328: 6e-6), and
the rounding of the result to bfloat16: half of a last place, 2^-8 of the value where its mantissa is 1: 2^-8 |y| + 1e-4 rms(y)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(y, x, w):
    want = x.double() @ w.double().t()
    assert y.dtype == torch.bfloat16 and y.shape == want.shape
    assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + 1e-4 * want.square().mean().sqrt()).all()


@pytest.mark.parametrize("m", [1, 2, 15, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("n,k", [(16, 64), (512, 576), (1040, 2816), (1024, 11328), (5632, 1024), (2064, 1984), (12288, 2816)])
def test_linear(m, n, k):
    """Waves without a step (K = 64), steps that do not divide by the waves or the split, row counts at the edges of the tiles."""
    from chronos import ops
    from chronos.ops import gemm as G

    plan = G.few_rows_plan(m, n, k)
    assert plan is not None or m > 1 and n * k > 7e6
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = (torch.randn(s, device=DEV, generator=g).bfloat16() for s in ((m, k), (n, k)))
    _check(ops.linear(x, w), x, w)
    if plan is not None:
        assert torch.equal(ops.linear(x.view(1, m, k), w)[0], G.pp_gemm(x, w, G.PP_PLAIN, plan)[0])


@pytest.mark.parametrize("cfg", [12, 13, 14, 15])
@pytest.mark.parametrize("splitk", [1, 2, 4, 8])
def test_uneven(cfg, splitk):
    from chronos import ops

    ops.load()
    m, n, k = {12: 32, 13: 64, 14: 16, 15: 16}[cfg], 96, 64 * (splitk * 11 + splitk // 2)
    g = torch.Generator(device=DEV).manual_seed(cfg)
    x, w = (torch.randn(s, device=DEV, generator=g).bfloat16() for s in ((m, k), (n, k)))
    for rows in (1, m - 1, m):
        _check(torch.ops.chronos.gemm_skinny(x[:rows], w, 0, cfg, splitk, None, None, 1e-5)[0], x[:rows], w)
    for bad in (lambda: torch.ops.chronos.gemm_skinny(x, w[:, :k - 8].contiguous(), 0, cfg, splitk, None, None, 1e-5),
                lambda: torch.ops.chronos.gemm_skinny(x, w, 1, cfg, splitk, None, None, 1e-5),
                lambda: torch.ops.chronos.gemm_skinny(torch.cat([x, x[:1]]), w, 0, cfg, splitk, None, None, 1e-5)):
        with pytest.raises(RuntimeError):
            bad()


def test_other_operands():
    """What the kernels do not take goes where it went: strided and misaligned operands, other types, gradients."""
    from chronos import ops

    g = torch.Generator(device=DEV).manual_seed(3)
    big = torch.randn(40, 1100, device=DEV, generator=g).bfloat16()
    w = torch.randn(256, 1024, device=DEV, generator=g).bfloat16()
    _check(ops.linear(big[:8, 3:1027], w), big[:8, 3:1027], w)
    flat = torch.randn(8 * 1024 + 1, device=DEV, generator=g).bfloat16()[1:].view(8, 1024)
    _check(ops.linear(flat, w), flat, w)
    wt = torch.randn(1024, 256, device=DEV, generator=g).bfloat16().t()
    _check(ops.linear(big[:8, :1024].contiguous(), wt), big[:8, :1024], wt)
    xf = torch.randn(8, 1024, device=DEV, generator=g)
    assert ops.linear(xf, w.float()).dtype == torch.float32
    xg = big[:8, :1024].contiguous().requires_grad_()
    ops.linear(xg, w).float().sum().backward()
    assert xg.grad is not None and xg.grad.shape == xg.shape
    ys = torch.vmap(lambda r: ops.linear(r, w))(big[:8, :1024].contiguous())
    _check(ys, big[:8, :1024], w)


@pytest.mark.parametrize("m", [2, 16, 64])
def test_autocast_and_subclasses(m):
    """Products that somebody has to see: under autocast they take its type, of a subclass they come back as one."""
    from chronos import ops
    from chronos.ops import gemm as G

    class Marked(torch.Tensor):
        pass

    x, w = (torch.randn(s, device=DEV).bfloat16() for s in ((m, 1024), (1024, 1024)))
    assert G.few_rows_plan(m, 1024, 1024) is not None
    with torch.autocast("cuda", torch.float16):
        y = ops.linear(x, w)
        assert y.dtype == torch.float16 and torch.equal(y, torch.matmul(x, w.t()))
    assert ops.linear(x, w).dtype == torch.bfloat16
    assert type(ops.linear(x, w.as_subclass(Marked))) is Marked
