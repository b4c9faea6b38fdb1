"""gemm_slab.hip: a workgroup's walk over its tiles (whole rounds, halves in the last one, one slab per tile), partial tiles in both
directions, and the epilogues of the hybrid decoders against float32."""
import pytest
import torch

DEV = "cuda"
pytestmark = pytest.mark.gpu


def _operands(m, n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
    return x, (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(torch.bfloat16)


def _close(y, ref):
    """One rounding to bfloat16 (2^-9 of the value) on top of float32 sums, whose order may move a value by 2^-20 of the operands."""
    err = (y.float() - ref).abs() - ref.abs() * 2.0 ** -8
    assert err.max().item() < 1e-4 * max(1.0, ref.abs().max().item())


@pytest.mark.parametrize("tiles", [1, 127, 128, 129, 255, 256, 257, 384, 385, 513, 800, 1100])
@pytest.mark.parametrize("k", [64, 192])
def test_every_tile_once(tiles, k):
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    m = 256 * tiles - 5     # one column of W tiles, the last x tile partial
    x, w = _operands(m, 256, k, tiles + k)
    y, _ = G.pp_gemm(x, w, G.PP_PLAIN, (88, 1))
    _close(y, x.float() @ w.float().t())


@pytest.mark.parametrize("m,n", [(585, 11264), (641, 11264), (128, 65536), (100, 65540), (300, 21760), (300, 22016), (256 * 256 + 5, 256),
                                 (256 * 300 + 77, 512), (256 * 300 + 129, 512), (1025, 8192), (2400, 7168)])
@pytest.mark.parametrize("k", [64, 128, 320])
def test_last_rows_as_halves(m, n, k):
    """x tiles of at most 128 rows at the end are one half each where one round of halves holds them and what whole rounds leave, at
    and past that line."""
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    x, w = _operands(m, n, k, m + n + k)
    ref = x.float() @ w.float().t()
    y, _ = G.pp_gemm(x, w, G.PP_PLAIN, (88, 1))
    _close(y, ref)
    g, u = ref[:, : n // 2], ref[:, n // 2:]
    if n % 256 == 0:
        _close(torch.ops.chronos.gemm_act(x, w, 3, float("inf"), 1.0, 1.0), g * torch.sigmoid(g) * (u + 1))


@pytest.mark.parametrize("m,n,k", [(1, 256, 64), (300, 512, 128), (2446, 5632, 192), (4100, 20224, 64)])
@pytest.mark.parametrize("limit,slope,shift", [(float("inf"), 1.0, 0.0), (0.75, 1.702, 1.0)])
def test_gated_unit(m, n, k, limit, slope, shift):
    from chronos import ops

    ops.load()
    x, w = _operands(m, n, k, m + n)
    h = x.float() @ w.float().t()
    g, u = h[:, : n // 2].clamp(max=limit), h[:, n // 2:].clamp(-limit, limit)
    _close(torch.ops.chronos.gemm_act(x, w, 3, limit, slope, shift), g * torch.sigmoid(slope * g) * (u + shift))


@pytest.mark.parametrize("m,n,k", [(1, 4, 64), (257, 1032, 128), (4100, 8196, 64)])
@pytest.mark.parametrize("mode", [4, 5])
def test_activation(m, n, k, mode):
    from chronos import ops

    ops.load()
    x, w = _operands(m, n, k, m + n + mode)
    h = x.float() @ w.float().t()
    ref = h.relu() ** 2 if mode == 4 else torch.nn.functional.gelu(h)
    _close(torch.ops.chronos.gemm_act(x, w, mode, 0.0, 0.0, 0.0), ref)


@pytest.mark.parametrize("m,n,k,s", [(1, 4, 128, 2), (129, 260, 192, 3), (585, 2048, 5632, 4), (384, 4096, 1024, 8), (300, 1032, 704, 11),
                                     (1100, 1024, 1024, 16), (2047, 2048, 256, 4), (70, 4096, 14336, 16)])
def test_slices_of_k(m, n, k, s):
    """Tiles and halves over slices of K, plain, with the residual's epilogue, and the same bits again in a graph's replays."""
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    x, w = _operands(m, n, k, m + n + k)
    ref = x.float() @ w.float().t()
    y, _ = G.pp_gemm(x, w, G.PP_PLAIN, (88, s))
    _close(y, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y2, _ = G.pp_gemm(x, w, G.PP_PLAIN, (88, s))
    for _ in range(3):
        y2.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y2, y)
    if n % 256 == 0:
        res = torch.randn(m, n, device=DEV).to(torch.bfloat16)
        z, part = G.pp_gemm(x, w, G.PP_RESID, (88, s), resid=res)
        assert torch.equal(z, y + res)
        want = z.double().square().view(m, n // 128, 128).sum(-1)
        assert ((part.double() - want).abs() <= want * 128 * 2.0 ** -24).all()


# x tiles of 128, 160, 192, 224 and 256 rows (80 tiles of W rows; their first and last row counts), two rounds of 160, whole rounds with halves
# behind, and the same with two slices of K
@pytest.mark.parametrize("m", [5, 384, 385, 480, 481, 576, 577, 672, 673, 768, 769, 960, 1300])
@pytest.mark.parametrize("k,s", [(64, 1), (192, 1), (384, 2)])
def test_rows_of_a_tile(m, k, s):
    """Every epilogue against float32, and every row the same bits as among other rows, where tiles have another height."""
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    n = 20480 // s
    x, w = _operands(m, n, k, m + k)
    ref = x.float() @ w.float().t()
    y, _ = G.pp_gemm(x, w, G.PP_PLAIN, (88, s))
    _close(y, ref)
    cut = m // 3 + 1
    assert torch.equal(torch.cat([G.pp_gemm(v.contiguous(), w, G.PP_PLAIN, (88, s))[0] for v in (x[:cut], x[cut:])]), y)
    res = torch.randn(m, n, device=DEV).to(torch.bfloat16)
    z, part = G.pp_gemm(x, w, G.PP_RESID, (88, s), resid=res)
    assert torch.equal(z, y + res)
    want = z.double().square().view(m, n // 128, 128).sum(-1)
    assert ((part.double() - want).abs() <= want * 128 * 2.0 ** -24).all()
    if s == 1:
        g, u = ref[:, : n // 2], ref[:, n // 2:]
        _close(torch.ops.chronos.gemm_act(x, w, 3, 1.5, 1.7, 1.0), g.clamp(max=1.5) * torch.sigmoid(1.7 * g.clamp(max=1.5)) * (u.clamp(-1.5, 1.5) + 1))
        sums = x.float().square().view(m, 32, -1).sum(-1).contiguous()
        scale = torch.rsqrt(x.float().square().mean(-1, keepdim=True) + 1e-5)
        _close(torch.ops.chronos.gemm_pp(x, w, 0, 88, 1, None, sums, 1e-5, False)[0], ref * scale)
