"""One token per sequence of the recurrences (csrc/hybrid/state_step.hip): every form against one step in float64, sequences without a token,
fresh ones, columns off the lanes' tiles.

Tolerance: float32 rounding, 2^-24 per operation, of sums over at most 256 rows: 2^-24 sqrt(256) = 1e-6 of the result's norm, taken twice."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
COUNT, STARTS, SLOTS = [1, 0, 1, 1, 1], [0, 3, 9, 1, 4], [2, 5, 0, 4, 1]


@pytest.mark.parametrize("form", ["fixed", "token", "rows", "delta", "delta_rows", "mlstm"])
@pytest.mark.parametrize("HK,H,D,Dv", [(2, 4, 32, 40), (2, 2, 64, 64), (1, 3, 128, 72), (4, 4, 128, 256), (2, 2, 256, 516)])
def test_step(form, HK, H, D, Dv):
    from chronos.ops import hybrid as hops

    if form == "mlstm":
        HK = H
    T = sum(COUNT)
    g = torch.Generator(device=DEV).manual_seed(H * D + Dv)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    rand = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    qs = [0]
    for n in COUNT:
        qs.append(qs[-1] + n)
    proj = rnd(T, 2 * HK * D + H * Dv + 12).bfloat16()
    S = rnd(7, H, D, Dv)
    S0, p = S.clone(), proj.double()
    q, k = (p[:, i * HK * D:(i + 1) * HK * D].view(T, HK, D) for i in (0, 1))
    v = p[:, 2 * HK * D:2 * HK * D + H * Dv].view(T, H, Dv)
    ranges = (i32(qs), i32(STARTS), i32(SLOTS))
    beta = vs = None
    if form == "mlstm":
        n, m, gp = rnd(7, H, D), rnd(7, H), rnd(T, 2 * H)
        n0, m0 = n.double(), m.double()
        o = hops.mlstm_scan(proj, gp, *ranges, S, n, m, H, D, Dv, 9.0, 1)
        ig, fg = 9 * torch.tanh(gp[:, :H].double() / 9), torch.nn.functional.logsigmoid(9 * torch.tanh(gp[:, H:].double() / 9))
    else:
        delta = form.startswith("delta")
        dec = rand(H) if form == "fixed" else rand(T, H, D) if form.endswith("rows") else rand(T, H)
        qsc, ksc = (rand(T, HK), rand(T, HK)) if form != "fixed" else (None, None)
        beta = rand(T, H) if delta else None
        vs = rand(T, H) if form == "token" else None
        o = hops.linear_scan(proj, 0, HK * D, 2 * HK * D, qsc, ksc, 0.3, dec, beta, *ranges, S, HK, H, D, Dv, vs, 1)
        q = q * (qsc.double()[..., None] if qsc is not None else 0.3)
        k = k * (ksc.double()[..., None] if ksc is not None else 1.0)
        d = dec.double().expand(T, H) if dec.dim() < 3 else dec.double()
    q, k = q.repeat_interleave(H // HK, 1), k.repeat_interleave(H // HK, 1)
    want, Sw = torch.empty(T, H, Dv, dtype=torch.double, device=DEV), S0.double()
    for b, cnt in enumerate(COUNT):
        if not cnt:
            continue
        t, sl, keep = qs[b], SLOTS[b], float(STARTS[b] > 0)
        s = Sw[sl] * keep
        if form == "mlstm":
            mn = torch.maximum(fg[t] + m0[sl] * keep, ig[t])
            a, w = torch.exp(fg[t] + m0[sl] * keep - mn), torch.exp(ig[t] - mn)
            s = a[:, None, None] * s + (w[:, None] * k[t])[:, :, None] * v[t][:, None]
            nn = a[:, None] * n0[sl] * keep + w[:, None] * k[t]
            qt = q[t] * D ** -0.5
            want[t] = (qt[:, None] @ s)[:, 0] / (torch.maximum((nn * qt).sum(-1).abs(), torch.exp(-mn)) + 1e-6)[:, None]
        else:
            s = d[t].view(H, -1, 1) * s
            u = v[t] * (vs[t].double()[:, None] if vs is not None else 1.0)
            if beta is not None:
                u = beta[t].double()[:, None] * (u - (k[t][:, None] @ s)[:, 0])
            s = s + k[t][:, :, None] * u[:, None]
            want[t] = (q[t][:, None] @ s)[:, 0]
        Sw[sl] = s
    assert float((o.double() - want).norm() / want.norm()) < 2e-6
    assert float((S.double() - Sw).norm() / Sw.norm()) < 2e-6
    assert torch.equal(S[3], S0[3]) and torch.equal(S[5], S0[5]) and torch.equal(S[6], S0[6])


@pytest.mark.parametrize("count", [[3, 0, 0], [0, 2, 0, 1], [2, 5, 0]])
@pytest.mark.parametrize("max_q", [0, 1])
@pytest.mark.parametrize("form", ["fixed", "token", "rows", "delta", "mlstm"])
def test_longer_ranges(form, max_q, count):
    """Ranges of several tokens where the launch takes one per sequence for the longest: beside empty ones when nobody says (T <= B),
    or with a hint of 1.  Against the plain recurrence of hybrid_ref in float32."""
    from chronos.ops import hybrid as hops

    H, D, Dv, T = 2, 64, 72, sum(count)
    g = torch.Generator().manual_seed(T)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    qs = [sum(count[:i]) for i in range(len(count) + 1)]
    args = [rnd(T, 2 * H * D + H * Dv + 16).bfloat16(), *(i32(x) for x in (qs, [4, 0, 7, 2][:len(count)], [1, 3, 0, 4][:len(count)])), rnd(5, H, D, Dv)]
    n, m, gp = rnd(5, H, D), rnd(5, H), rnd(T, 2 * H)
    dec = torch.rand(H, generator=g) if form == "fixed" else torch.rand(T, H, D, generator=g) if form == "rows" else torch.rand(T, H, generator=g)
    beta = torch.rand(T, H, generator=g) if form == "delta" else None

    def run(dev):
        proj, q, p0, sl, S = (t.to(dev, copy=True) for t in args)
        if form == "mlstm":
            st = [S, n.to(dev, copy=True), m.to(dev, copy=True)]
            return hops.mlstm_scan(proj, gp.to(dev), q, p0, sl, *st, H, D, Dv, 9.0, max_q), *st
        o = hops.linear_scan(proj, 0, H * D, 2 * H * D, None, None, 0.3, dec.to(dev), None if beta is None else beta.to(dev), q, p0, sl, S,
                             H, H, D, Dv, None, max_q)
        return o, S

    for got, want in zip(run(DEV), run("cpu")):   # both sides round
        assert float((got.cpu() - want).norm() / want.norm()) < 4e-6


@pytest.mark.parametrize("form", ["fixed", "token", "rows", "delta", "delta_rows", "mlstm"])
@pytest.mark.parametrize("HK,H,D,Dv", [(2, 4, 32, 100), (4, 4, 256, 128), (2, 4, 64, 264), (4, 4, 128, 132), (2, 4, 256, 512)])
def test_many_rows(form, HK, H, D, Dv):
    """Launches with a workgroup for every CU: 32 and 64 lanes to a row of the state (columns in 128s and 256s), two of 66 sequences empty.
    Every sequence is one step, all of them at once in float64; tolerance as above."""
    from chronos.ops import hybrid as hops

    if form == "mlstm":
        HK = H
    B, g = 66, torch.Generator(device=DEV).manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    rand = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    count = torch.ones(B, dtype=torch.int64)
    count[[5, 60]] = 0
    T, rep = int(count.sum()), H // HK
    assert T * H * ((Dv + 255) // 256) >= 256
    qs = torch.cat([torch.zeros(1, dtype=torch.int64), count.cumsum(0)]).int().to(DEV)
    start, slots = torch.arange(B, device=DEV).int() % 3, torch.randperm(B + 2, device=DEV, generator=g)[:B].int()
    live = count.bool().to(DEV)
    sl, keep = slots[live].long(), (start[live] > 0).double()[:, None]
    proj, S = rnd(T, 2 * HK * D + H * Dv + 12).bfloat16(), rnd(B + 2, H, D, Dv)
    S0, p = S.clone(), proj.double()
    q, k = (p[:, i * HK * D:(i + 1) * HK * D].view(T, HK, D) for i in (0, 1))
    v = p[:, 2 * HK * D:2 * HK * D + H * Dv].view(T, H, Dv)
    s = S0[sl].double() * keep[..., None, None]
    if form == "mlstm":
        n, m, gp = rnd(B + 2, H, D), rnd(B + 2, H), rnd(T, 2 * H)
        n0, m0 = n[sl].double() * keep[..., None], m[sl].double() * keep
        o = hops.mlstm_scan(proj, gp, qs, start, slots, S, n, m, H, D, Dv, 9.0, 1)
        ig, fg = 9 * torch.tanh(gp[:, :H].double() / 9), torch.nn.functional.logsigmoid(9 * torch.tanh(gp[:, H:].double() / 9))
        mn = torch.maximum(fg + m0, ig)
        a, w = torch.exp(fg + m0 - mn), torch.exp(ig - mn)
        s = a[..., None, None] * s + (w[..., None] * k)[..., None] * v[:, :, None]
        nn = a[..., None] * n0 + w[..., None] * k
        den = torch.maximum((nn * q * D ** -0.5).sum(-1).abs(), torch.exp(-mn)) + 1e-6
        # (before the division: a denominator that nearly cancels magnifies its own rounding)
        got, want = o.double() * den[..., None], (q[:, :, None] @ s)[:, :, 0] * D ** -0.5
        assert float((n[sl].double() - nn).norm() / nn.norm()) < 2e-6 and float((m[sl].double() - mn).norm() / mn.norm()) < 2e-6
    else:
        delta = form.startswith("delta")
        dec = rand(H) if form == "fixed" else rand(T, H, D) if form.endswith("rows") else rand(T, H)
        qsc, ksc = (rand(T, HK), rand(T, HK)) if form != "fixed" else (None, None)
        beta, vs = rand(T, H) if delta else None, rand(T, H) if form == "token" else None
        o = hops.linear_scan(proj, 0, HK * D, 2 * HK * D, qsc, ksc, 0.3, dec, beta, qs, start, slots, S, HK, H, D, Dv, vs, 1)
        q = (q * (qsc.double()[..., None] if qsc is not None else 0.3)).repeat_interleave(rep, 1)
        k = (k * (ksc.double()[..., None] if ksc is not None else 1.0)).repeat_interleave(rep, 1)
        s = (dec.double().expand(T, H) if dec.dim() < 3 else dec.double()).reshape(T, H, -1, 1) * s
        u = v * (vs.double()[..., None] if vs is not None else 1.0)
        if delta:
            u = beta.double()[..., None] * (u - (k[:, :, None] @ s)[:, :, 0])
        s = s + k[..., None] * u[:, :, None]
        got, want = o.double(), (q[:, :, None] @ s)[:, :, 0]
    assert float((got - want).norm() / want.norm()) < (1e-5 if form == "mlstm" else 2e-6)
    assert float((S[sl].double() - s).norm() / s.norm()) < 2e-6
    rest = torch.ones(B + 2, dtype=torch.bool, device=DEV)
    rest[sl] = False
    assert torch.equal(S[rest], S0[rest])
