"""Joins that take a product as the float32 slices of its split: the same bits as from the summed and rounded product."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


@pytest.mark.parametrize("rows,d", [(1, 1024), (3, 1032), (64, 2048), (5, 2056), (17, 4096), (2, 4104), (64, 8192)])
@pytest.mark.parametrize("S", [1, 2, 5, 8, 16])
def test_joins(rows, d, S):
    from chronos.ops import hybrid as hops

    g = torch.Generator(device=DEV).manual_seed(rows + d + S)
    ys = torch.randn(S, rows, d, device=DEV, generator=g)
    y = ys[0].clone()
    for k in range(1, S):
        y += ys[k]
    y, x0, w = y.to(BF), torch.randn(rows, d, device=DEV, generator=g), torch.randn(d, device=DEV, generator=g)
    for join in (lambda a, x: hops.add_layer_norm(a, x, w, 1e-5, BF), lambda a, x: hops.scale_add_rms_norm(a, x, w, 1.7, 1e-6, BF)):
        x1, x2 = x0.clone(), x0.clone()
        h1, h2 = join(ys, x1), join(y, x2)
        # the row's statistics are summed over other lanes in another order: d rounded additions at most, 2^-24 each
        tol = d * 2.0 ** -24
        assert ((x1 - x2).abs() <= tol * (x2.abs() + 4 * w.abs())).all() and h1.dtype == BF and h1.shape == h2.shape
        assert torch.equal(h1, x1.to(BF))


@pytest.mark.parametrize("m,n,k", [(1, 1024, 2816), (16, 1024, 2816), (64, 1024, 4096), (8, 2048, 8192), (40, 4096, 14336), (64, 4096, 8192)])
def test_products(m, n, k):
    from chronos import ops
    from chronos.ops import gemm as G, hybrid as hops

    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(BF), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)
    ys = hops.matmul_slices(x, w)
    assert ys.dim() == 3 and ys.shape[0] == G.few_rows_plan(m, n, k)[1] and ys.shape[1:] == (m, n)
    y = ys[0].clone()
    for s in ys[1:]:
        y += s
    assert torch.equal(y.to(BF), ops.linear(x, w))


def test_what_has_no_slices():
    from chronos.ops import hybrid as hops

    x, w = torch.randn(16, 2816, device=DEV).to(BF), torch.randn(1024, 2816, device=DEV).to(BF)
    assert hops.matmul_slices(x, w).dim() == 3
    for a, b in ((x.view(2, 8, 2816), w), (torch.randn(128, 2816, device=DEV).to(BF), w), (x[:, :1024].contiguous(), w[:, :1024].contiguous()),
                 (x, w.clone().requires_grad_(True)), (x.float(), w.float())):
        assert hops.matmul_slices(a, b).dtype == a.dtype
    with torch.autocast("cuda", torch.bfloat16):
        assert hops.matmul_slices(x, w).dtype == BF
    x0 = torch.randn(16, 1024, device=DEV)
    for bad in (torch.randn(2, 16, 1020, device=DEV), torch.randn(2, 15, 1024, device=DEV), torch.randn(65, 16, 1024, device=DEV)):
        with pytest.raises(RuntimeError):
            hops.add_layer_norm(bad, x0, torch.ones(1024, device=DEV), 1e-5, BF)
