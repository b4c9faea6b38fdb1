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
