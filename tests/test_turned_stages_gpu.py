"""Tiles that take K round from a place of their own: gemm_lg.hip's ring tiles of one x tile (stages), moe_grouped.hip's over large weights (k-steps).  Every stage
is taken once, whatever their number."""
import pytest
import torch

DEV = "cuda"
pytestmark = pytest.mark.gpu

# ring tiles of at most 128 x rows whose pieces fill their waves, and those of 256 rows; 14, 18 and 12 take K in 32s
RING = [(72, (2, 8, 9, 32)), (74, (2, 7, 31)), (75, (16, 31)), (79, (5, 32)), (38, (33, 64)), (39, (8, 64)), (32, (65, 128)), (19, (100,)), (15, (128,)), (29, (40, 128)),
        (30, (129, 256)), (35, (200,)), (14, (137,)), (18, (256,)), (12, (250,))]


def _operands(m, n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return g, torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).to(torch.bfloat16)


# stages per slice (K / 64 / split): 64, 65, one, 9 (more and fewer than rings of 4 to 12 hold), 11, 43, 172; N: a part tile, ragged, more workgroups than stages
@pytest.mark.parametrize("cfg,rows", RING)
@pytest.mark.parametrize("k,split", [(4096, 1), (4160, 1), (4096, 64), (4608, 8), (5632, 8), (11008, 4), (11008, 1)])
@pytest.mark.parametrize("n", [16, 4100, 20004])
def test_turned_products(cfg, rows, k, split, n):
    from chronos import ops

    ops.load()
    for m in rows:
        _, x, w = _operands(m, n, k, cfg + k + n)
        want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        # float32 sums of exact products in any order: half a last place of the largest partial sum for each of k terms
        if cfg in (72, 74, 75, 79, 38, 39, 32, 19):
            y = torch.ops.chronos.gemm_slices(x, w, cfg, split, False)
            assert ((y.double().sum(0) - want).abs() <= size * k * 2 ** -24).all()
        if split == 1:
            y, _ = torch.ops.chronos.gemm_pp(x, w, 0, cfg, 1, None, None, 1e-5, False)
            assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + size * k * 2 ** -24).all()


@pytest.mark.parametrize("cfg,rows", RING)
@pytest.mark.parametrize("k", [4096, 4672])
def test_turned_epilogues(cfg, rows, k):
    """Gated units behind a folded norm, and residuals with their partial sums: as in order but for last bits of the sums."""
    from chronos import ops

    ops.load()
    n = 1536
    for m in rows:
        g, x, w = _operands(m, n, k, cfg + m)
        r = torch.randn(m, n, device=DEV, generator=g).to(torch.bfloat16)
        part = (x.float() ** 2).view(m, 64, -1).sum(-1)
        for mode, res, pt in ((1, None, part), (0, None, part), (2, r, None)):
            a, b = (torch.ops.chronos.gemm_pp(x, w, mode, cfg, 1, res, pt, 1e-5, False, in_order) for in_order in (False, True))
            # sums of variance 1: float32 orders move them by less than 2e-5 (a sum with a normal number, a gated unit: 3 times that), so that values are the same or, where
            # the sum lies that close to a boundary, a bfloat16 step apart, at most 2^-7 of the value.  Gated units round gate, sigmoid's product and up number: a step
            # (2^-8 to 2^-7) of each, the gate's times the unit's relative slope 1 + g (1 - sigmoid(g)), 5 at g = -6: 8 steps of 2^-8 in all.  A residual's product is rounded by itself
            # before the sum (of at most |r| + |sum|)
            d, mag = (a[0].float() - b[0].float()).abs(), torch.maximum(a[0].float().abs(), b[0].float().abs())
            mag = 4 * mag if mode == 1 else mag if mode == 0 else 2 * mag + r.float().abs()
            assert (d <= mag * 2 ** -7 + 6e-5).all() and float((d > 0).float().mean()) < 0.05
            if mode == 2:
                assert ((a[1] - b[1]).abs() <= 0.02 * b[1].abs() + 1e-3).all()


@pytest.mark.parametrize("cfg,rows", [(74, (2, 8)), (72, (3, 8, 30)), (38, (64,))])
def test_sums_in_order(cfg, rows):
    """in_order: a product's rows have the bits of the same rows among 128 on a kernel that is never turned (several x tiles); without it they are turned."""
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    _, x, w = _operands(128, 28672, 4096, cfg)
    all_rows = G.pp_gemm(x, w, 0, (cfg, 1))[0]
    for m in rows:
        xs = x[:m].contiguous()
        assert torch.equal(G.pp_gemm(xs, w, 0, (cfg, 1), in_order=True)[0], all_rows[:m])
        assert not torch.equal(G.pp_gemm(xs, w, 0, (cfg, 1))[0], all_rows[:m])


# k-steps of the two products: 2 and 256 (fewer and more than the ring holds), 30 and 32.  Batches of tiles of 32, 64, 128 and (not of 128 wide ones) 256 rows, placed in
# the first product and by a launch, on both sides of where the chosen experts' weights are 256 MB
@pytest.mark.parametrize("form", ["gelu", "glu"])
@pytest.mark.parametrize("d,F", [(128, 16384), (1920, 2048)])
def test_turned_experts(d, F, form):
    """moe_grouped.hip's tiles over experts' weights of 256 MB and more, against the PyTorch reference (tolerance of the other expert tests), and a
    token's result whatever else is in the batch."""
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    E, top, bf, T = 80, 8, torch.bfloat16, 4000
    assert E * F * d * 2 >= 1 << 28
    g = torch.Generator(device=DEV).manual_seed(T + d)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    h, wt = rnd(T, d).to(bf), torch.rand(T, top, device=DEV, generator=g)
    idx = torch.rand(T, E, device=DEV, generator=g).topk(top, -1).indices.int()
    wu, wd = (rnd(E, F * (2 if form == "glu" else 1), d) * d ** -0.5).to(bf), (rnd(E, d, F) * F ** -0.5).to(bf)
    if form == "glu":
        order = hops.moe_glu_row_order(F).to(DEV)
        tiled = wu[:, order].contiguous()
        run = lambda n: hops.moe_glu_ffn(h[:n].contiguous(), idx[:n].contiguous(), wt[:n].contiguous(), tiled, wd, 7.0, 1.702, 1.0, bf, True)  # noqa: E731
        want = ref.moe_glu_ffn(h[:200], idx[:200], wt[:200], wu, wd, 7.0, 1.702, 1.0, bf).float()
    else:
        run = lambda n: hops.moe_ffn(h[:n].contiguous(), idx[:n].contiguous(), wt[:n].contiguous(), wu, wd, 1, bf)  # noqa: E731
        want = ref.moe_ffn(h[:200], idx[:200], wt[:200], wu, wd, 1, bf).float()
    whole = run(T)
    assert (whole[:200].float() - want).abs().max() <= 1.5e-2 * want.abs().max()
    for n in (1, 2, 3, 9, 10, 60, 130, 300, 450, 900, 1800, 2500):
        assert torch.equal(run(n), whole[:n]), n
