"""Experts for few tokens: projection and choice in one launch, placing inside the first grouped product."""
import pytest
import torch

from chronos.ops import hybrid as hops, hybrid_ref as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(*s, seed=0):
    return torch.randn(*s, generator=torch.Generator().manual_seed(seed)).to(DEV)


# outputs around a wave's share (16) and the most that one launch takes (64), widths around its runs of 512 columns, tokens around 256
@pytest.mark.parametrize("n", [2, 16, 17, 48, 63, 64, 65])
@pytest.mark.parametrize("d", [8, 504, 512, 520, 1024, 1536, 4096, 4104])
@pytest.mark.parametrize("t", [1, 5, 256, 257])
def test_route(n, d, t):
    h, w = _rand(t, d).bfloat16(), (_rand(n, d, seed=1) * 2 * d ** -0.5).bfloat16()
    b, top = _rand(n, seed=2) * 0.01, min(4, n)
    groups = 4 if n % 4 == 0 and n >= 16 else 1
    for got, want in ((hops.moe_route(h, w, b, top), ref.moe_route(h, w, b, top)), (hops.moe_route_topk(h, w, b, top), ref.moe_route_topk(h, w, b, top)),
                      (hops.moe_route_group(h, w, top, groups, max(1, groups // 2), 2.5), ref.moe_route_group(h, w, top, groups, max(1, groups // 2), 2.5))):
        same = got[0].long() == want[0].long()
        # float32 sums of d products differ in their order: choices between logits that close may differ, one in a thousand at most
        assert same.float().mean() > 0.999 - 1.0 / same.numel() * (same.numel() < 1000)
        assert ((got[1] - want[1]).abs() * same).max() < 2e-5


def _ffn(t, top, e, skew, form, d, f):
    g = torch.Generator().manual_seed(t)
    idx = torch.stack([torch.randperm(e + 2, generator=g)[:top] for _ in range(t)]) if e + 2 >= top else torch.zeros(t, top)
    if skew == "one":
        idx[:] = e - 1
    if skew == "holes":
        idx[::3] = -1
    idx = idx.int().to(DEV)
    h, wt = _rand(t, d).bfloat16(), torch.rand(t, top, generator=g).to(DEV)
    up, dn = (_rand(e, 2 * f if form == "glu" else f, d, seed=3) * d ** -0.5).bfloat16(), (_rand(e, d, f, seed=4) * f ** -0.5).bfloat16()
    real = idx.clone()
    if form == "glu":
        y = hops.moe_glu_ffn(h, idx, wt, up[:, hops.moe_glu_row_order(f).to(DEV)].contiguous(), dn, 7.0, 1.702, 1.0, torch.bfloat16, True)
    else:
        y = hops.moe_ffn(h, idx, wt, up, dn, hops.ACT_GELU, torch.bfloat16)
    # the sum over a token's choices in float64
    want = torch.zeros(t, d, dtype=torch.float64, device=DEV)
    hd = h.double()
    for k in range(top):
        for x in real[:, k].unique().tolist():
            rows = real[:, k] == x
            if x < 0 or (x >= e and form == "glu"):
                continue
            if x >= e:
                v = hd[rows]
            else:
                u = hd[rows] @ up[x].double().t()
                if form == "glu":
                    a, b = u[:, :f].clamp(max=7.0), u[:, f:].clamp(-7.0, 7.0)
                    u = a * torch.sigmoid(1.702 * a) * (b + 1.0)
                else:
                    u = torch.nn.functional.gelu(u)
                v = u @ dn[x].double().t()
            want[rows] += v * wt[rows, k].double()[:, None]
    # three roundings to bfloat16 on the way (products, activation, rows) and one of the sum: 2^-9 each
    assert (y.double() - want).norm() <= 2 ** -7 * want.norm() + 1e-12


# items around a run of 64 and the most that place themselves (512), up to 64 experts; skewed: all items one expert's, several tiles
@pytest.mark.parametrize("t,top,e", [(1, 1, 1), (1, 4, 64), (31, 2, 8), (33, 2, 8), (16, 4, 64), (127, 4, 32), (128, 4, 64), (129, 4, 64), (64, 2, 65)])
@pytest.mark.parametrize("skew", ["even", "one", "holes"])
@pytest.mark.parametrize("form", ["gelu", "glu"])
def test_ffn(t, top, e, skew, form):
    _ffn(t, top, e, skew, form, 128, 128)


# weights around what one product marks as read once (256 MB of the experts that can be chosen), with and without placing in the launch
@pytest.mark.parametrize("t,top,e,d,f", [(3, 2, 8, 4096, 4096), (4, 2, 8, 4096, 4096), (4, 2, 8, 4096, 3968), (300, 2, 40, 2048, 2048)])
def test_ffn_read_once(t, top, e, d, f):
    _ffn(t, top, e, "even", "gelu", d, f)


# tokens per expert at the lines between tiles of 32, 64 and 128 rows, for experts that make few workgroups and more
@pytest.mark.parametrize("t,top,e,d", [(288, 2, 8, 128), (289, 2, 8, 128), (1280, 2, 8, 128), (1281, 2, 8, 128), (512, 4, 64, 256), (513, 4, 64, 256), (1408, 4, 64, 256), (1409, 4, 64, 256),
                                       (480, 4, 96, 512), (481, 4, 96, 512), (1728, 4, 96, 512), (1729, 4, 96, 512)])
@pytest.mark.parametrize("skew", ["even", "one", "holes"])
@pytest.mark.parametrize("form", ["gelu", "glu"])
def test_ffn_tiles(t, top, e, d, skew, form):
    _ffn(t, top, e, skew, form, d, d)
