"""Reductions across lanes (csrc/include/chronos_hip.h): a wave's sum, maximum and best value end in every lane, whichever lane holds what."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d", [256, 512, 1024, 4096])
def test_every_column_counts(d):
    """One large entry per row, in every column in turn: a norm that loses or repeats a lane is off by it."""
    from chronos.ops import hybrid as hops

    hops.load()
    x = torch.full((d, d), 1e-3, device=DEV)
    x.fill_diagonal_(1.0)
    got = hops.rms_norm(x.clone(), torch.ones(d, device=DEV), 1e-6, torch.float32)
    xd = x.double()
    want = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-6)
    # sums of at most 4096 like terms: a few roundings of 2^-24 each side of the root
    assert float(((got.double() - want).abs() / want).max()) < 2e-6


@pytest.mark.parametrize("n,top", [(1, 1), (16, 4), (63, 3), (64, 8), (65, 8), (256, 8)])
def test_every_expert_is_found(n, top):
    """Choices whose largest values lie at every number in turn, equal ones in the order of their numbers."""
    from chronos.ops import hybrid as hops

    hops.load()
    d = 256
    h = torch.zeros(n, d, device=DEV, dtype=torch.bfloat16)
    h[torch.arange(n), torch.arange(n)] = 1.0
    w = torch.zeros(n, d, device=DEV, dtype=torch.bfloat16)   # token t: expert t 3, all others 1
    w[:, :n] = 1.0
    w[torch.arange(n), torch.arange(n)] = 3.0
    idx, wt = hops.moe_route_topk(h, w, torch.zeros(n, device=DEV), top)
    for t, row in enumerate(idx.tolist()):
        assert row == [t] + [e for e in range(n) if e != t][:top - 1]
    assert torch.equal(wt[:, 0], wt[:1, 0].expand(n)) and bool((wt[:, 1:] == wt[:1, 1:]).all())
