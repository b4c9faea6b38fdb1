"""Projections between few and many rows that no measured plan lists (ops/gemm.py mid_rows_plan) against the float64 product of the same bfloat16
operands: float32 sums (2^-24 sqrt(K) of the result's root mean square, K <= 11264: 7e-6) and one rounding to bfloat16 (2^-9 of the value, 2^-8 where the
mantissa is 1)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    return torch.randn(m, k, device=DEV, generator=g).bfloat16(), torch.randn(n, k, device=DEV, generator=g).bfloat16()


def _check(y, x, w, tol=2 ** -8):
    want = x.double() @ w.double().t()
    assert ((y.double() - want).abs() <= want.abs() * tol + 1e-5 * want.square().mean().sqrt()).all()


# rows at the edges of the rule and of the tiles, outputs that end inside a tile, K of one, two and odd numbers of steps per slice
@pytest.mark.parametrize("m", [33, 63, 64, 65, 96, 127, 128, 129, 255, 257, 511, 512])
@pytest.mark.parametrize("n,k", [(512, 512), (528, 11264), (1040, 576), (1024, 2816), (4112, 4096), (12288, 1024), (12304, 2048), (32768, 512), (16400, 4096)])
def test_linear(m, n, k):
    from chronos import ops
    from chronos.ops import gemm as G

    x, w = _operands(m, n, k)
    y = ops.linear(x, w)
    _check(y, x, w)
    assert torch.equal(y, ops.linear(x.view(1, m, k), w)[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = ops.linear(x, w)
    for _ in range(3):
        z.fill_(float("nan"))
        torch.randn(1 << 16, device=DEV).sum().item()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, y)
    if m <= 64 and n >= 12288:
        f = G.product_f32(x, w)
        if f is not None:
            _check(f, x, w, 0.0)


def test_other_operands():
    """What the kernels do not take goes where it went: strides, types, gradients, an output tensor."""
    from chronos import ops

    x, w = _operands(100, 1024, 1024)
    _check(ops.linear(x[:, :512], w[:, :512]), x[:, :512], w[:, :512])
    _check(ops.linear(x[:, 3:515].contiguous(), w[:, 3:515].contiguous()), x[:, 3:515], w[:, 3:515])
    assert ops.linear(x.float(), w.float()).dtype == torch.float32
    out = torch.empty(100, 1024, device=DEV, dtype=torch.bfloat16)
    assert ops.linear(x, w, out=out).data_ptr() == out.data_ptr()
    _check(out, x, w)
    xg = x.clone().requires_grad_()
    ops.linear(xg, w).float().sum().backward()
    want = w.float().sum(0)
    assert ((xg.grad.float() - want).abs() <= 2 ** -7 * want.abs() + 0.05 * want.abs().mean()).all()


# what slab_rows_plan takes from the library or from whole K: two to eight slices, ragged rows and outputs
@pytest.mark.parametrize("m,n,k", [(300, 4096, 8192), (1100, 4096, 11008), (1500, 4096, 11008), (2100, 2048, 5632), (2446, 4096, 4096), (1089, 3656, 8192), (1100, 4096, 14336)])
def test_slab_rows(m, n, k):
    from chronos import ops
    from chronos.ops import gemm as G

    plan = G.slab_rows_plan(m, n, k)
    assert plan is not None and plan[0] == 88 and plan != G.many_rows_plan(m, n, k)
    x, w = _operands(m, n, k)
    y = ops.linear(x, w)
    _check(y, x, w)
    assert torch.equal(y, G.pp_gemm(x, w, G.PP_PLAIN, plan)[0])
