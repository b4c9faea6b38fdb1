"""Gated linear attention's chunks with their tiles made ahead (csrc/hybrid/gla_scan.hip gla_walk_kernel) against the chunks that make them between the
steps, which a call takes whose longest range is said to be one chunk: the same terms, their products in another order, so both are within a
float32 sum's roundings of each other."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# ranges of no token, one, a chunk, one more; many sequences (more than a wave finds at once); heads that share keys; columns off the slabs.  odd: decays that
# leave the range, then NaN among the keys, infinite and large values
@pytest.mark.parametrize("lens,HK,H,D,Dv", [([100, 1, 17, 16, 33, 0, 2, 15], 2, 6, 64, 72), ([200, 31, 32], 4, 4, 32, 64),
                                            ([47, 48, 81], 4, 8, 128, 200), ([255], 16, 16, 128, 256), ([64, 130], 2, 2, 256, 72),
                                            ([(37 * i) % 97 for i in range(70)], 2, 2, 128, 64), ([0, 0, 90, 0], 16, 16, 128, 128), ([700, 65], 2, 2, 128, 64)])
@pytest.mark.parametrize("odd", [0, 1, 2])
def test_both_forms(lens, HK, H, D, Dv, odd):
    from chronos.ops import hybrid as hops

    hops.load()
    T, B = sum(lens), len(lens)
    for longest in (16, max(lens)):
        assert torch.ops.chronos.hy_chunk_scan_pays(3, T, B, H, D, Dv, longest)
    g = torch.Generator(device=DEV).manual_seed(T + D)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    rand = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    y = rnd(T, 2 * HK * D + H * Dv).bfloat16()
    decay = rand(T, H, D) ** (1 / 16)
    if odd:
        decay[3::50], decay[9::31], decay[11::37], decay[20::29], decay[23::61, :, ::3] = 0.0, 1e-30, 1.0, -0.8, 1.4
    if odd == 2:
        y[T // 2, -1], y[T // 3, -2], y[T // 4, HK * D + 3], y[T // 5, -3] = float("nan"), float("inf"), float("nan"), 1e12
    qs, ks, vs = rand(T, HK), rand(T, HK), rand(T, H)
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    S0, got = rnd(B + 1, H, D, Dv) * 0.3, []
    for longest in (16, max(lens)):
        S = S0.clone()
        o = hops.linear_scan(y, 0, HK * D, 2 * HK * D, qs, ks, 1.0, decay, None, i32(start), i32([7 * (b % 2) for b in range(B)]), i32(list(range(1, B + 1))),
                             S, HK, H, D, Dv, vs, longest)
        got.append((o, S))
    for a, b in zip(*got):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
        a, b = (t.double().where(t.isfinite(), torch.zeros((), dtype=torch.double, device=DEV)) for t in (a, b))
        # by (head, column), over the tokens or the states' rows (a single token's read-out may be next to nothing beside its terms; the large values are a
        # column's own): sums of D + 16 terms, each rounded once, at random: sqrt(272) 2^-24
        over = (0,) if a.dim() == 3 else (0, 2)
        assert bool(((a - b).norm(dim=over) <= 1e-6 * b.norm(dim=over)).all())
    assert bool(got[0][0].isnan().any()) == (odd == 2)
