"""The ring tiles' and the GEMV's epilogues with more to do (gemm_ring, gemv_act): float32 outputs of a few rows behind the product's, activations."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16
CONFIGS = [(72, (9, 32)), (74, (2, 33)), (75, (31,)), (79, (32,)), (38, (64, 65)), (39, (1, 64, 200)), (32, (127, 128)), (19, (100, 129))]


def _operands(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    return g, torch.randn(m, k, device=DEV, generator=g).to(BF), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(BF)


@pytest.mark.parametrize("cfg,ms", CONFIGS)
@pytest.mark.parametrize("n0,nf,k", [(4, 1, 64), (128, 16, 320), (1020, 13, 512), (4096, 64, 4096)])
@pytest.mark.parametrize("split", [1, 4])
def test_rows_behind(cfg, ms, n0, nf, k, split):
    from chronos import ops

    ops.load()
    if k // 64 % split:
        return
    for m in ms:
        g, x, w = _operands(m, n0 + -(-nf // 32) * 32, k)
        for bias in (None, torch.randn(nf, device=DEV, generator=g)):
            y, yf = torch.ops.chronos.gemm_ring(x, w, cfg, split, 0, n0, nf, bias, 0.0, 0.0, 0.0)
            want = x.double() @ w.double().t()
            size = (x.double().abs() @ w.double().abs().t()) * k * 2 ** -24          # float32 sums in any order
            assert y.shape == (m, n0) and yf.shape == (m, nf) and yf.dtype == torch.float32
            assert ((y.double() - want[:, :n0]).abs() <= want[:, :n0].abs() * 2 ** -8 + size[:, :n0]).all()
            wf = want[:, n0:n0 + nf] + (0 if bias is None else bias.double())
            assert ((yf.double() - wf).abs() <= size[:, n0:n0 + nf] + wf.abs() * 2 ** -23).all()


@pytest.mark.parametrize("cfg,ms", CONFIGS + [(0, (1,))])      # (0: the GEMV)
@pytest.mark.parametrize("n,k", [(128, 512), (2176, 1024), (14336, 4096)])
@pytest.mark.parametrize("mode", [3, 4, 5])
def test_activations(cfg, ms, n, k, mode):
    """float32 sums move a value by less than 2e-5 (sums of products of variance 1 / K; slopes below 3), and there is one rounding to bfloat16."""
    from chronos import ops

    ops.load()
    for m in ms:
        _, x, w = _operands(m, n, k)
        h, F = x.double() @ w.double().t(), n // 2
        for limit, slope, shift in ((float("inf"), 1.0, 0.0), (0.75, 1.702, 1.0)) if mode == 3 else ((0.0, 0.0, 0.0),):
            if cfg:
                y = torch.ops.chronos.gemm_ring(x, w, cfg, 1, mode, 0, 0, None, limit, slope, shift)[0]
            else:
                y = torch.ops.chronos.gemv_act(x, w, mode, limit, slope, shift)
            a, u = h[:, :F].clamp(max=limit), h[:, F:].clamp(-limit, limit)
            want = a * torch.sigmoid(slope * a) * (u + shift) if mode == 3 else h.relu() ** 2 if mode == 4 else torch.nn.functional.gelu(h)
            size = torch.maximum(h[:, :F].abs(), h[:, F:].abs()) if mode == 3 else h.abs()
            assert y.dtype == BF and y.shape == want.shape
            assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + 2e-5 * size.clamp(min=1)).all()


@pytest.mark.parametrize("m,n,k,mode,takes", [(1, 22016, 4096, 3, True), (64, 14336, 4096, 4, True), (40, 22016, 4096, 3, True), (100, 5632, 1024, 3, True),
                                              (64, 5632, 1024, 3, False), (32, 11264, 2048, 3, True), (5, 16384, 1024, 4, True)])
def test_which_products(m, n, k, mode, takes):
    from chronos.ops import gemm as G

    _, x, w = _operands(m, n, k)
    assert (G.product_act(x, w, mode, 7.0, 1.702, 1.0) is not None) == takes
    joined = torch.cat([w, w[:32]])
    assert (G.product_rows(x, joined, n, 16, None) is not None) == (m > 1 or n * k < 30e6)


@pytest.mark.parametrize("m", [8, 100, 400])
@pytest.mark.parametrize("rows,n0,nf", [(1030, 1024, 6), (1029, 1024, 5), (1031, 1024, 6)])
def test_joined_without_padding(m, rows, n0, nf):
    """matmul_rowdot of a joined matrix that ends with its last row."""
    from chronos.ops import hybrid as hops

    hops.load()
    g, x, w = _operands(m, rows, 1024)
    bias = torch.randn(nf, device=DEV, generator=g)
    y, yf = hops.matmul_rowdot(x, w[:n0], w[n0:n0 + nf].contiguous(), bias, (w, n0, nf))
    want = x.double() @ w[:n0 + nf].double().t()
    size = (x.double().abs() @ w[:n0 + nf].double().abs().t()) * 1024 * 2 ** -24          # float32 sums in any order
    assert ((y.double() - want[:, :n0]).abs() <= want[:, :n0].abs() * 2 ** -8 + size[:, :n0]).all()
    assert ((yf.double() - want[:, n0:] - bias.double()).abs() <= size[:, n0:] + 2 ** -22 * (want[:, n0:].abs() + bias.abs())).all()


@pytest.mark.parametrize("bad", [dict(cfg=36), dict(mode=3, n=130), dict(mode=4, split=2), dict(n0=2), dict(nf=0), dict(n0=128, nf=40), dict(split=5), dict(mode=2)])
def test_what_is_refused(bad):
    from chronos import ops

    ops.load()
    mode = bad.get("mode", 0)
    _, x, w = _operands(8, bad.get("n", 160), 256)
    n0, nf = (bad.get("n0", 128), bad.get("nf", 16)) if mode == 0 else (0, 0)
    with pytest.raises(RuntimeError):
        torch.ops.chronos.gemm_ring(x, w, bad.get("cfg", 39), bad.get("split", 1), mode, n0, nf, None, 1.0, 1.0, 0.0)
