"""Projection and choice of many tokens in one launch (csrc/hybrid/moe.hip moe_route_tile_kernel), against the same tokens in calls of up to 512, which
project and choose in two."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one expert, whole and broken tiles of 16, the most and one more (two launches); the last workgroup's tokens whole, broken, one
@pytest.mark.parametrize("T,d,N,top", [(513, 64, 1, 1), (528, 256, 16, 4), (700, 1024, 17, 2), (1025, 2048, 32, 8), (2000, 4096, 24, 6), (5000, 512, 33, 4)])
@pytest.mark.parametrize("form", ["softmax", "topk", "groups"])
def test_like_two_launches(T, d, N, top, form):
    from chronos.ops import hybrid as hops

    hops.load()
    g = torch.Generator(device=DEV).manual_seed(T + N)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    h, w, b = rnd(T, d).bfloat16(), (rnd(N, d) * 2 * d ** -0.5).bfloat16(), rnd(N) * 0.1
    h[5] = h[3]          # equal tokens, and one with equal logits throughout
    h[7] = 0.0
    ng = 4 if N % 4 == 0 else 1

    def route(x):
        if form == "softmax":
            return hops.moe_route(x, w, b * 0.01, top)
        if form == "topk":
            return hops.moe_route_topk(x, w, b, top)
        return hops.moe_route_group(x, w, top, ng, max(1, ng - 1), 1.5)

    idx, wt = route(h)
    parts = [route(h[i:i + 500]) for i in range(0, T, 500)]
    want, wwant = (torch.cat(p) for p in zip(*parts))
    same = (idx == want).all(dim=1)
    # logits of another order of sums: a few roundings of 2^-24 apart, which few choices among random ones turn on
    assert float((~same).float().mean()) < 2e-3 and bool(same[7]) and torch.equal(idx[5], idx[3])
    assert float((wt[same] - wwant[same]).abs().max()) < 1e-5
    assert int(idx.min()) >= 0 and int(idx.max()) < N


@pytest.mark.parametrize("T,d,N,top", [(513, 64, 1, 1), (4999, 1024, 16, 16), (700, 320, 17, 17), (8191, 2048, 32, 32)])
def test_logits_are_the_projections(T, d, N, top):
    """The choices follow from the logits that the projection by itself gives, ties and near ties included: not one differs."""
    from chronos.ops import hybrid as hops

    hops.load()
    g = torch.Generator(device=DEV).manual_seed(T - N)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    h, w, b = rnd(T, d).bfloat16(), (rnd(N, d) * 0.02 * d ** -0.5).bfloat16(), rnd(N) * 0.02
    if N > 4:
        w[3], b[3] = w[1], b[1]
    z = hops.rowdot(h, w, b)
    val, want = torch.sort(z, dim=1, descending=True, stable=True)   # (equal ones: the lower row first)
    idx, wt = hops.moe_route_topk(h, w, b, top)
    assert torch.equal(idx.long(), want[:, :top])
    # exponentials of float32 differences, N of them added up and divided by: N + 4 roundings of 2^-24 and expf's two
    assert float((wt.double() - torch.softmax(val[:, :top].double(), 1)).abs().max()) < (N + 8) * 2.0 ** -24
