"""Joins that take a product of more than 64 rows as the float32 slices of its split: the bits of the summed and rounded product."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


# the rules' two kernels: 64-row ring tiles (part tiles of rows), the slab walk (part rows; whole tiles)
@pytest.mark.parametrize("m,n,k,cfg", [(65, 1024, 2816, 39), (200, 2048, 2048, 39), (400, 1024, 4096, 39), (200, 4096, 11008, 88), (1351, 2048, 8192, 88),
                                       (768, 4096, 14336, 88)])
def test_products(m, n, k, cfg):
    from chronos import ops
    from chronos.ops import gemm as G, hybrid as hops

    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(BF), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)
    ys = hops.matmul_parts(x, w)
    assert G._linear_plan(m, n, k) == (cfg, ys.shape[0]) and ys.shape[1:] == (m, n) and ys.dtype == torch.float32
    y = ys[0].clone()
    for s in ys[1:]:
        y += s
    assert torch.equal(y.to(BF), ops.linear(x, w))
    x0, wn = torch.randn(m, n, device=DEV, generator=g), torch.randn(n, device=DEV, generator=g)
    for join in (lambda a, r: hops.add_layer_norm(a, r, wn, 1e-5, BF), lambda a, r: hops.scale_add_rms_norm(a, r, wn, 1.7, 1e-6, BF)):
        r1, r2 = x0.clone(), x0.clone()
        h1, _ = join(ys, r1), join(y.to(BF), r2)
        # a row's statistics are summed over other lanes: d rounded additions at most, 2^-24 each
        assert ((r1 - r2).abs() <= n * 2.0 ** -24 * (r2.abs() + 4 * wn.abs())).all() and torch.equal(h1, r1.to(BF))


def test_what_has_no_parts():
    from chronos.ops import hybrid as hops

    x, w = torch.randn(200, 2816, device=DEV).to(BF), torch.randn(1024, 2816, device=DEV).to(BF)
    assert hops.matmul_parts(x, w).dim() == 3
    for a, b in ((x.view(2, 100, 2816), w), (x[:, :1024].contiguous(), w[:, :1024].contiguous()), (x, w.clone().requires_grad_(True)), (x.float(), w.float()),
                 (torch.randn(8192, 2816, device=DEV).to(BF), w)):
        assert hops.matmul_parts(a, b).dtype == a.dtype
    with torch.autocast("cuda", torch.bfloat16):
        assert hops.matmul_parts(x, w).dtype == BF
    with pytest.raises(RuntimeError):
        torch.ops.chronos.gemm_slices(x, w, 88, 1, False)     # (one slice of the slab walk is its plain product)


@pytest.mark.parametrize("m,n,k", [(16, 1024, 2816), (200, 1024, 2816), (1, 1024, 1024)])
def test_weight_off_the_16_bytes(m, n, k):
    """A norm's weight that lies behind others in one buffer: joins took it with a product's rows, and do with its slices and in the product behind them."""
    from chronos.ops import hybrid as hops

    hops.load()
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x, w = torch.randn(m, k, device=DEV, generator=g).to(BF), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)
    flat = torch.randn(n + 1, device=DEV, generator=g)
    x0, off, on = torch.randn(m, n, device=DEV, generator=g), flat[1:], flat[1:].clone()
    assert off.data_ptr() % 16 == 4
    y = hops.matmul_parts(x, w)
    assert (y.dim() == 3) == (m > 1)
    if m > 1:   # (slices: one kernel for both)
        for join in (lambda r, v: hops.add_layer_norm(y, r, v, 1e-5, BF), lambda r, v: hops.scale_add_rms_norm(y, r, v, 1.7, 1e-6, BF)):
            r1, r2 = x0.clone(), x0.clone()
            assert torch.equal(join(r1, off), join(r2, on)) and torch.equal(r1, r2)
    else:
        got = [hops.JoinedRows(y, x0.clone(), v, 1.7, 1e-6) for v in (off, on)]
        a, b = (j.product(w, 1)[0] for j in got)
        assert torch.equal(a, b) and torch.equal(got[0].stream(), got[1].stream())
