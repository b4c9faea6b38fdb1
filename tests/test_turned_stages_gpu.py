"""gemm_lg.hip's ring tiles of one x tile, whose workgroups start their K at different stages: every stage is taken once, whatever their number."""
import pytest
import torch

DEV = "cuda"
pytestmark = pytest.mark.gpu


# stages per slice (K / 64 / split): one, fewer than the ring holds, as many, one more, odd, many; N: a part tile, one round, more workgroups than
# stages on every XCD, ragged
@pytest.mark.parametrize("cfg,rows", [(72, (9, 32)), (75, (16, 31)), (79, (32,)), (38, (33, 64)), (39, (64,)), (32, (65, 128)), (19, (100,)), (15, (128,)), (29, (40, 128))])
@pytest.mark.parametrize("k,split", [(64, 1), (192, 1), (512, 2), (576, 1), (832, 1), (4096, 1)])
@pytest.mark.parametrize("n", [16, 4100, 70656])
def test_turned_products(cfg, rows, k, split, n):
    from chronos import ops

    ops.load()
    g = torch.Generator(device=DEV).manual_seed(cfg + k + n)
    w = torch.randn(n, k, device=DEV, generator=g).to(torch.bfloat16)
    for m in rows:
        x = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
        want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        # float32 sums of exact products in any order: half a last place of the largest partial sum for each of k terms
        if cfg in (72, 75, 79, 38, 39, 32, 19):
            y = torch.ops.chronos.gemm_slices(x, w, cfg, split, False)
            assert ((y.double().sum(0) - want).abs() <= size * k * 2 ** -24).all()
        if split == 1 and n % 4 == 0:
            y, _ = torch.ops.chronos.gemm_pp(x, w, 0, cfg, 1, None, None, 1e-5, False)
            assert ((y.double() - want).abs() <= want.abs() * 2 ** -8 + size * k * 2 ** -24).all()


@pytest.mark.parametrize("cfg,rows", [(74, (2, 8)), (72, (3, 8))])
def test_sums_of_up_to_eight_rows_keep_their_order(cfg, rows):
    """A layer's product of up to 8 rows has the bits of the same rows among 64 on a kernel that is not turned (two x tiles)."""
    from chronos import ops

    ops.load()
    g = torch.Generator(device=DEV).manual_seed(cfg)
    w = torch.randn(28672, 4096, device=DEV, generator=g).to(torch.bfloat16)
    x = torch.randn(64, 4096, device=DEV, generator=g).to(torch.bfloat16)
    all_rows, _ = torch.ops.chronos.gemm_pp(x, w, 0, cfg, 1, None, None, 1e-5, False)
    for m in rows:
        y, _ = torch.ops.chronos.gemm_pp(x[:m].contiguous(), w, 0, cfg, 1, None, None, 1e-5, False)
        assert torch.equal(y, all_rows[:m])


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
