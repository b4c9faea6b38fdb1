"""The delta rule's chunks with their tiles made ahead (csrc/hybrid/chunk_scan.hip delta_tiles_kernel): the bits of the chunks that make them between
the steps, which a call takes whose longest range is said to be one chunk."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# ranges of no token, one, a tile, a chunk, one more; many sequences (more than a wave finds at once); heads that share keys; columns off the slabs
@pytest.mark.parametrize("lens,HK,H,D,Dv", [([300, 1, 65, 64, 129, 0, 2, 33], 2, 6, 64, 72), ([200, 63, 128], 4, 4, 32, 64),
                                            ([191, 192, 193], 4, 8, 128, 200), ([1000], 8, 8, 128, 128),
                                            ([(37 * i) % 131 for i in range(70)], 2, 2, 128, 64), ([0, 0, 66, 0], 16, 16, 128, 128)])
@pytest.mark.parametrize("nan", [False, True])
def test_same_bits(lens, HK, H, D, Dv, nan):
    from chronos.ops import hybrid as hops

    hops.load()
    T, B = sum(lens), len(lens)
    for longest in (64, max(lens)):
        assert torch.ops.chronos.hy_chunk_scan_pays(2, T, B, H, D, Dv, longest)
    g = torch.Generator(device=DEV).manual_seed(T + D)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    y = rnd(T, 2 * HK * D + H * Dv).bfloat16()
    ks = y[:, HK * D:2 * HK * D].float().view(T, HK, D).norm(dim=-1).reciprocal()
    qs, beta = torch.rand(T, HK, device=DEV, generator=g), torch.rand(T, H, device=DEV, generator=g)
    decay = torch.exp(-2 * torch.rand(T, H, device=DEV, generator=g))
    decay[3::50], decay[9::31], decay[11::37], decay[20::29], decay[23::61] = 0.0, 1e-30, 1.0, -0.8, 1.4
    if nan:
        y[T // 2, -1] = float("nan")
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    S0, got = rnd(B + 1, H, D, Dv) * 0.3, []
    for longest in (64, max(lens)):
        S = S0.clone()
        o = hops.linear_scan(y, 0, HK * D, 2 * HK * D, qs, ks, 1.0, decay, beta, i32(start), i32([7 * (b % 2) for b in range(B)]), i32(list(range(1, B + 1))),
                             S, HK, H, D, Dv, max_q=longest)
        got.append((o, S))
    bits = lambda t: t.contiguous().view(torch.int32)  # noqa: E731
    assert all(torch.equal(bits(a), bits(b)) for a, b in zip(*got))
    assert bool(got[0][0].isnan().any()) == nan
