"""Recurrent mixers of decode rows in one launch (csrc/hybrid/state_mix.hip) against the launches they stand for, which their own tests check against
float64; sequences without a token, fresh ones, ranges longer than the launch was told, column counts off the lanes' tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
STARTS, SLOTS = [0, 3, 9, 1, 4], [2, 5, 0, 4, 1]


def _setup(count, HK, H, D, Dv, extra, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    qs = [0]
    for n in count:
        qs.append(qs[-1] + n)
    C = 2 * HK * D + H * Dv
    proj = rnd(qs[-1], C + H * Dv + extra).bfloat16()
    tok = i32([b for b, n in enumerate(count) for _ in range(n)])
    return rnd, proj, C, tok, (i32(qs), i32(STARTS), i32(SLOTS))


def _close(a, b, tol):
    assert a.shape == b.shape and a.dtype == b.dtype
    assert float((a.double() - b.double()).norm()) <= tol * float(b.double().norm()) + 1e-12


# bfloat16 results: the launches round q, k and v between convolution and state (2^-9 each, relative; up to 4 of them reach an output) and
# the result once more; float32 states see the first of these, or (rows, gates: no rounding between) float32 sums in another order
@pytest.mark.parametrize("count", [[1, 0, 1, 1, 1], [3, 0, 2, 1, 6]])
@pytest.mark.parametrize("HK,H,D,Dv", [(2, 4, 64, 40), (2, 2, 64, 64), (1, 2, 128, 128), (3, 3, 128, 72), (2, 4, 128, 256), (2, 2, 256, 132),
                                      (8, 16, 128, 128), (13, 13, 128, 128), (12, 12, 128, 128)])   # (states from 4 MB on: read as data used once)
def test_delta(count, HK, H, D, Dv):
    from chronos.ops import hybrid as hops

    rnd, proj, C, tok, rng = _setup(count, HK, H, D, Dv, 4, H * D + Dv)
    taps, ab, a_log, w = rnd(C, 4) * 0.5, rnd(proj.shape[0], 2 * H), rnd(H) * 0.3, rnd(H * Dv)
    hist, S = rnd(7, 3, C).bfloat16(), rnd(7, H, D, Dv) * 0.3
    assert hops.one_step_ok(proj, 1, D, Dv, H // HK, S, hist, taps, w) and not hops.one_step_ok(proj, 2, D, Dv, H // HK, S)
    h1, S1 = hist.clone(), S.clone()
    y = hops.short_conv(proj, taps, tok, *rng, h1, True, max_q=0)
    sc = hops.delta_prep(y, ab, a_log, HK, H, D, D ** -0.5)
    o = hops.linear_scan(y, 0, HK * D, 2 * HK * D, sc[0], sc[1], 1.0, sc[2], sc[3], *rng, S1, HK, H, D, Dv, max_q=0)
    want = hops.head_norm_gate(o, proj, C, w, 1e-6, True, torch.bfloat16)
    got = hops.delta_step(proj, taps, ab, a_log, *rng, hist, S, HK, H, D, Dv, D ** -0.5, C, w, 1e-6)
    assert torch.equal(hist, h1)
    _close(S, S1, 4 * 2.0 ** -9)
    _close(got, want, 5 * 2.0 ** -9)
    assert torch.equal(S[3], S1[3]) and torch.equal(S[6], S1[6])


@pytest.mark.parametrize("count", [[1, 0, 1, 1, 1], [3, 0, 2, 1, 6]])
@pytest.mark.parametrize("H,D,Dv,R", [(2, 64, 40, 16), (4, 128, 256, 16), (3, 128, 72, 7), (2, 256, 132, 1), (7, 128, 256, 16)])
def test_rows(count, H, D, Dv, R):
    from chronos.ops import hybrid as hops

    rnd, proj, C, tok, rng = _setup(count, H, H, D, Dv, 8, H * D + Dv)
    low, w2, b2, w, S = rnd(proj.shape[0], R), rnd(R, H * D), rnd(H * D) + 2, rnd(H * Dv), rnd(7, H, D, Dv) * 0.3
    S1 = S.clone()
    dec = hops.low_rank_decay(low, w2, b2, 1 / 16)
    o = hops.linear_scan(proj, 0, H * D, 2 * H * D, None, None, D ** -0.5, dec, None, *rng, S1, H, H, D, Dv, max_q=0)
    want = hops.head_norm_gate(o, proj, C, w, 1e-6, True, torch.bfloat16)
    got = hops.rows_step(proj, low, w2, b2, 1 / 16, *rng, S, H, D, Dv, D ** -0.5, C, w, 1e-6)
    _close(S, S1, 2e-6)
    _close(got, want, 2.0 ** -9)


@pytest.mark.parametrize("count", [[1, 0, 1, 1, 1], [3, 0, 2, 1, 6]])
@pytest.mark.parametrize("H,D,Dv", [(2, 64, 40), (4, 128, 256), (3, 128, 72), (2, 256, 132), (5, 256, 192)])
def test_gates(count, H, D, Dv):
    from chronos.ops import hybrid as hops

    rnd, proj, C, tok, rng = _setup(count, H, H, D, Dv, 8, H * D + Dv)
    gp, w, S, n, m = rnd(proj.shape[0], 2 * H), rnd(H * Dv), rnd(7, H, D, Dv) * 0.3, rnd(7, H, D), rnd(7, H)
    S1, n1, m1 = S.clone(), n.clone(), m.clone()
    o = hops.mlstm_scan(proj, gp, *rng, S1, n1, m1, H, D, Dv, 9.0, 0)
    want = hops.mlstm_out(o, proj, C, w, 1e-6, torch.bfloat16)
    got = hops.mlstm_step(proj, gp, *rng, S, n, m, H, D, Dv, 9.0, C, w, 1e-6)
    for a, b in ((S, S1), (n, n1), (m, m1)):
        _close(a, b, 2e-6)
    _close(got, want, 2.0 ** -9)
