"""The chunked forms of the linear-state recurrences (csrc/hybrid/chunk_scan.hip) against the token-by-token recurrence in
float64, at the edges of a chunk (64 tokens) and of its 16-token tiles, with ranges that continue a state, with decays of 0
and 1, negative ones and ones above 1, and with column counts off the 64-column slabs.

Tolerance: inputs are exact in both (bfloat16 and float32); what differs is float32 rounding, 2^-24 per operation, of
sums over at most 129 tokens and 256 state rows and of one exponential per token.  Errors of independent roundings grow with the
square root of their number: sqrt(129 * 256) * 2^-24 = 1.1e-5 at the very worst alignment of the result's cancellation,
2e-6 over a whole result's norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS, STARTS, SLOTS = [1, 64, 129, 0, 17, 63, 65, 16], [0, 5, 0, 3, 9, 0, 2, 7], [2, 0, 4, 1, 3, 7, 5, 8]


def _setup(seed, T, C, H, D, Dv):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    qs = [0]
    for n in LENS:
        qs.append(qs[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    return g, rnd, qs, (i32(qs), i32(STARTS), i32(SLOTS))


def _in_chunks(form, lens, H, D, Dv, longest=None):
    """These launches do go in chunks."""
    from chronos.ops import hybrid as hops

    hops.load()
    assert torch.ops.chronos.hy_chunk_scan_pays({"mlstm": 1, "delta": 2, "rows": 3}.get(form, 0), sum(lens), len(lens), H, D, Dv, longest or max(lens))


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("HK,H,D,Dv,form", [(2, 4, 32, 40, "token"), (1, 2, 64, 64, "token"), (2, 2, 128, 72, "head"),
                                            (1, 3, 256, 128, "token"), (4, 4, 128, 128, "head")])
def test_plain(HK, H, D, Dv, form):
    from chronos.ops import hybrid as hops

    _in_chunks("plain", LENS, H, D, Dv, sum(LENS) - len(LENS) + 1)   # (the bound that the op takes without max_q)
    T = sum(LENS)
    C = 2 * HK * D + H * Dv + 16
    g, rnd, qs, ranges = _setup(H * D + Dv, T, C, H, D, Dv)
    proj = rnd(T, C).bfloat16()
    if form == "head":
        decay, vs = 1 - torch.rand(H, device=DEV, generator=g) ** 4, None
        decay[0] = 1.0
    else:
        decay, vs = torch.exp(-2 * torch.rand(T, H, device=DEV, generator=g)), torch.rand(T, H, device=DEV, generator=g)
        decay[3::50], decay[9::31], decay[11::37], decay[20::29], decay[23::61] = 0.0, 1e-30, 1.0, -0.8, 1.4
    qsc, ksc = torch.rand(T, HK, device=DEV, generator=g), torch.rand(T, HK, device=DEV, generator=g)
    S = rnd(9, H, D, Dv) * 0.3
    S0 = S.clone()
    o = hops.linear_scan(proj, 8, 8 + HK * D, 8 + 2 * HK * D, qsc, ksc, 1.0, decay, None, *ranges, S, HK, H, D, Dv, vs)
    p = proj.double()
    q = (p[:, 8:8 + HK * D].view(T, HK, D) * qsc.double()[..., None]).repeat_interleave(H // HK, 1)
    k = (p[:, 8 + HK * D:8 + 2 * HK * D].view(T, HK, D) * ksc.double()[..., None]).repeat_interleave(H // HK, 1)
    v = p[:, 8 + 2 * HK * D:8 + 2 * HK * D + H * Dv].view(T, H, Dv) * (vs.double()[..., None] if vs is not None else 1.0)
    dec = decay.double().expand(T, H)
    want, Sw = torch.empty(T, H, Dv, dtype=torch.double, device=DEV), S0.double()
    for b, n in enumerate(LENS):
        s = torch.zeros(H, D, Dv, dtype=torch.double, device=DEV) if STARTS[b] == 0 else Sw[SLOTS[b]]
        for t in range(qs[b], qs[b] + n):
            s = dec[t][:, None, None] * s + k[t][:, :, None] * v[t][:, None]
            want[t] = (q[t][:, None] @ s)[:, 0]
        if n:
            Sw[SLOTS[b]] = s
    assert _rel(o, want) < 2e-6 and _rel(S, Sw) < 2e-6
    assert torch.equal(S[1], S0[1]) and torch.equal(S[6], S0[6]), "slots without tokens must stay untouched"


@pytest.mark.parametrize("HK,H,D,Dv,scales", [(2, 4, 32, 40, True), (1, 2, 64, 64, False), (3, 3, 128, 72, True), (2, 2, 256, 128, False)])
def test_rows(HK, H, D, Dv, scales):
    """One decay per state row (csrc/hybrid/gla_scan.hip, 16 tokens at a time, chunks whose products of decays leave the range token by
    token: the first sequences have some of both, the last two none)."""
    from chronos.ops import hybrid as hops

    _in_chunks("rows", LENS, H, D, Dv)
    T = sum(LENS)
    C = 2 * HK * D + H * Dv + 16
    g, rnd, qs, ranges = _setup(H * D + Dv, T, C, H, D, Dv)
    proj = rnd(T, C).bfloat16()
    rand = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    decay = rand(T, H, D) ** (1 / 8)
    decay[3:200:50], decay[9:200:31], decay[11::37], decay[20::29], decay[23::61, :, ::3] = 0.0, 1e-30, 1.0, -0.8, 1.4
    qsc, ksc, vs = (rand(T, HK), rand(T, HK), rand(T, H)) if scales else (None, None, None)
    S = rnd(9, H, D, Dv) * 0.3
    S0 = S.clone()
    o = hops.linear_scan(proj, 8, 8 + HK * D, 8 + 2 * HK * D, qsc, ksc, 0.7, decay, None, *ranges, S, HK, H, D, Dv, vs, max(LENS))
    p, one = proj.double(), torch.ones(T, 1, dtype=torch.double, device=DEV)
    q = (p[:, 8:8 + HK * D].view(T, HK, D) * (qsc.double()[..., None] if scales else 0.7)).repeat_interleave(H // HK, 1)
    k = (p[:, 8 + HK * D:8 + 2 * HK * D].view(T, HK, D) * (ksc.double() if scales else one)[..., None]).repeat_interleave(H // HK, 1)
    v = p[:, 8 + 2 * HK * D:8 + 2 * HK * D + H * Dv].view(T, H, Dv) * (vs.double() if scales else one)[..., None]
    want, Sw = torch.empty(T, H, Dv, dtype=torch.double, device=DEV), S0.double()
    for b, n in enumerate(LENS):
        s = torch.zeros(H, D, Dv, dtype=torch.double, device=DEV) if STARTS[b] == 0 else Sw[SLOTS[b]]
        for t in range(qs[b], qs[b] + n):
            s = decay[t].double()[..., None] * s + k[t][:, :, None] * v[t][:, None]
            want[t] = (q[t][:, None] @ s)[:, 0]
        if n:
            Sw[SLOTS[b]] = s
    assert _rel(o, want) < 2e-6 and _rel(S, Sw) < 2e-6
    assert torch.equal(S[1], S0[1]) and torch.equal(S[6], S0[6]), "slots without tokens must stay untouched"


@pytest.mark.parametrize("HK,H,D,Dv,form", [(2, 4, 32, 40, "token"), (2, 2, 64, 64, "head"), (2, 4, 128, 72, "token"), (1, 3, 128, 128, "same")])
def test_delta(HK, H, D, Dv, form):
    """The delta rule's 16-row solves: keys of length 1, in "same" all nearly one direction with betas near 1 (every token undoes
    most of the last one's write, the system is as far from the identity as it gets)."""
    from chronos.ops import hybrid as hops

    _in_chunks("delta", LENS, H, D, Dv)
    T = sum(LENS)
    C = 2 * HK * D + H * Dv + 16
    g, rnd, qs, ranges = _setup(H * D + Dv, T, C, H, D, Dv)
    proj = rnd(T, C)
    if form == "same":
        proj[:, 8 + HK * D:8 + 2 * HK * D] = 3 * rnd(HK * D) + 0.1 * proj[:, 8 + HK * D:8 + 2 * HK * D]
    proj = proj.bfloat16()
    beta = torch.rand(T, H, device=DEV, generator=g)
    if form == "same":
        beta = 1 - 0.05 * beta
    beta[5::23] = 0.0
    if form == "head":
        decay = 1 - torch.rand(H, device=DEV, generator=g) ** 4
        decay[0] = 1.0
    else:
        decay = torch.exp(-0.3 * torch.rand(T, H, device=DEV, generator=g))
        decay[3::50], decay[9::31], decay[11::37], decay[20::29], decay[23::61] = 0.0, 1e-30, 1.0, -0.8, 1.4
    p = proj.double()
    q, k = p[:, 8:8 + HK * D].view(T, HK, D), p[:, 8 + HK * D:8 + 2 * HK * D].view(T, HK, D)
    qsc, ksc = (1 / q.norm(dim=-1)).float(), (1 / k.norm(dim=-1)).float()
    S = rnd(9, H, D, Dv) * 0.3
    S0 = S.clone()
    o = hops.linear_scan(proj, 8, 8 + HK * D, 8 + 2 * HK * D, qsc, ksc, 1.0, decay, beta, *ranges, S, HK, H, D, Dv, max_q=max(LENS))
    q = (q * qsc.double()[..., None]).repeat_interleave(H // HK, 1)
    k = (k * ksc.double()[..., None]).repeat_interleave(H // HK, 1)
    v, dec, bt = p[:, 8 + 2 * HK * D:8 + 2 * HK * D + H * Dv].view(T, H, Dv), decay.double().expand(T, H), beta.double()
    want, Sw = torch.empty(T, H, Dv, dtype=torch.double, device=DEV), S0.double()
    for b, n in enumerate(LENS):
        s = torch.zeros(H, D, Dv, dtype=torch.double, device=DEV) if STARTS[b] == 0 else Sw[SLOTS[b]]
        for t in range(qs[b], qs[b] + n):
            s = dec[t][:, None, None] * s
            u = bt[t][:, None] * (v[t] - (k[t][:, None] @ s)[:, 0])
            s = s + k[t][:, :, None] * u[:, None]
            want[t] = (q[t][:, None] @ s)[:, 0]
        if n:
            Sw[SLOTS[b]] = s
    assert _rel(o, want) < 2e-6 and _rel(S, Sw) < 2e-6
    assert torch.equal(S[1], S0[1]) and torch.equal(S[6], S0[6]), "slots without tokens must stay untouched"


@pytest.mark.parametrize("H,D,Dv,gate", [(2, 32, 24, 1.0), (1, 64, 128, 6.0), (3, 128, 72, 1.0), (2, 256, 64, 4.0)])
def test_mlstm(H, D, Dv, gate):
    from chronos.ops import hybrid as hops

    _in_chunks("mlstm", LENS, H, D, Dv)
    T, cap = sum(LENS), 9.0
    C = 2 * H * D + 2 * H * Dv
    g, rnd, qs, ranges = _setup(H * D + Dv, T, C, H, D, Dv)
    proj, gp = rnd(T, C).bfloat16(), rnd(T, 2 * H) * gate
    gp[:, H:] += 2.0
    S, n, m = rnd(9, H, D, Dv) * 0.3, rnd(9, H, D) * 0.5, rnd(9, H)
    S0, n0, m0 = S.clone(), n.clone(), m.clone()
    o = hops.mlstm_scan(proj, gp, *ranges, S, n, m, H, D, Dv, cap, max(LENS))
    p, gd = proj.double(), gp.double()
    ig = cap * torch.tanh(gd[:, :H] / cap)
    fg = torch.nn.functional.logsigmoid(cap * torch.tanh(gd[:, H:] / cap))
    num, den = torch.empty(T, H, Dv, dtype=torch.double, device=DEV), torch.empty(T, H, dtype=torch.double, device=DEV)
    Sw, nw, mw = S0.double(), n0.double(), m0.double()
    for b, cnt in enumerate(LENS):
        s, nn, mm = (Sw[SLOTS[b]], nw[SLOTS[b]], mw[SLOTS[b]]) if STARTS[b] else (Sw[0] * 0, nw[0] * 0, mw[0] * 0)
        for t in range(qs[b], qs[b] + cnt):
            q, k = p[t, :H * D].view(H, D) * D ** -0.5, p[t, H * D:2 * H * D].view(H, D)
            v = p[t, 2 * H * D:2 * H * D + H * Dv].view(H, Dv)
            mn = torch.maximum(fg[t] + mm, ig[t])
            a, w, mm = torch.exp(fg[t] + mm - mn), torch.exp(ig[t] - mn), mn
            s = a[:, None, None] * s + (w[:, None] * k)[:, :, None] * v[:, None]
            nn = a[:, None] * nn + w[:, None] * k
            num[t] = (q[:, None] @ s)[:, 0]
            den[t] = torch.maximum((nn * q).sum(-1).abs(), torch.exp(-mm)) + 1e-6
        if cnt:
            Sw[SLOTS[b]], nw[SLOTS[b]], mw[SLOTS[b]] = s, nn, mm
    # a denominator that nearly cancels magnifies its own rounding: compare the read-out before the division
    assert _rel(o * den[..., None].float(), num) < 1e-5
    assert _rel(S, Sw) < 2e-6 and _rel(n, nw) < 2e-6 and _rel(m, mw) < 1e-6
    for t, t0 in ((S, S0), (n, n0), (m, m0)):
        assert torch.equal(t[1], t0[1]) and torch.equal(t[6], t0[6]), "slots without tokens must stay untouched"


@pytest.mark.parametrize("lens,starts", [([1100, 40, 0, 513, 1023], [0, 3, 5, 9, 0]), ([2500], [7])])
@pytest.mark.parametrize("form,D", [("token", 64), ("mlstm", 64), ("rows", 32), ("rows", 64), ("rows", 128), ("rows", 256)])
def test_segments(lens, starts, form, D):
    """Few, long sequences: their chunks are dealt to segments (1100 tokens: four of 18 chunks; 2500: ten of 40; one
    decay per row: nine of 69 and 16 of 157), whose states are carried first; against the same sequences in launches too wide for segments."""
    from chronos.ops import hybrid as hops

    H, Dv, T = 2, 72, sum(lens)
    _in_chunks(form, lens, H, D, Dv)
    _in_chunks(form, lens * 40, H, D, Dv)
    reps = 40   # copies of the sequences that fill the chip: no segments
    g = torch.Generator(device=DEV).manual_seed(T)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    proj, gp = rnd(T, 2 * H * D + 2 * H * Dv).bfloat16(), rnd(T, 2 * H)
    gp[:, H:] += 3.0
    dec = torch.exp(-0.2 * torch.rand(T, H, device=DEV, generator=g))
    dec[7::90], dec[11::400] = -0.9, 1.2
    if form == "rows":
        dec = torch.rand(T, H, D, device=DEV, generator=g) ** (1 / 16)
        dec[300:420:40], dec[7::90], dec[11::400], dec[23::610, :, ::3] = 0.0, -0.9, 1.2, 1e-30
    B = len(lens)
    S0, n0, m0 = rnd(B, H, D, Dv) * 0.3, rnd(B, H, D) * 0.5, rnd(B, H)

    def run(r):
        qs = [0]
        for n in lens * r:
            qs.append(qs[-1] + n)
        rg = (i32(qs), i32(starts * r), torch.arange(B * r, device=DEV).int())
        S, n, m = (t.repeat(r, *[1] * (t.dim() - 1)) for t in (S0, n0, m0))
        if form == "mlstm":
            o = hops.mlstm_scan(proj.repeat(r, 1), gp.repeat(r, 1), *rg, S, n, m, H, D, Dv, 9.0, max(lens))
        else:
            o = hops.linear_scan(proj.repeat(r, 1), 0, H * D, 2 * H * D, None, None, 0.3, dec.repeat(r, *[1] * (dec.dim() - 1)), None, *rg, S, H, H, D, Dv,
                                 None, max(lens))
        return o[:T], S[:B], n[:B], m[:B]

    a, w = run(1), run(reps)
    for x, y in zip(a[1:], w[1:]):
        assert _rel(x, y.double()) < 2e-6
    if form == "mlstm":   # (the read-out is divided by a sum that may nearly cancel: as in test_mlstm, before the division)
        den = _mlstm(proj, gp, S0, n0, m0, lens, starts, 9.0, False)[1][..., None]
        assert _rel(a[0] * den, w[0] * den) < 1e-5
    else:
        assert _rel(a[0], w[0].double()) < 2e-6


def _mlstm(proj, gp, S0, n0, m0, lens, starts, cap, whole=True):
    """(numerators, denominators, S, n, m) of the mlstm recurrence in float64; not ``whole``: without numerators and S."""
    B, H, D, Dv = S0.shape
    T, p, gd = proj.shape[0], proj.double(), gp.double()
    ig, fg = cap * torch.tanh(gd[:, :H] / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(gd[:, H:] / cap))
    q, k = p[:, :H * D].view(T, H, D) * D ** -0.5, p[:, H * D:2 * H * D].view(T, H, D)
    v = p[:, 2 * H * D:2 * H * D + H * Dv].view(T, H, Dv)
    num, den = torch.zeros(T, H, Dv, dtype=torch.double, device=DEV), torch.empty(T, H, dtype=torch.double, device=DEV)
    S, n, m = S0.double(), n0.double(), m0.double()
    t = 0
    for b, cnt in enumerate(lens):
        keep = float(starts[b] > 0)
        s, nn, mm = S[b] * keep, n[b] * keep, m[b] * keep
        for t in range(t, t + cnt):
            mn = torch.maximum(fg[t] + mm, ig[t])
            a, w, mm = torch.exp(fg[t] + mm - mn), torch.exp(ig[t] - mn), mn
            nn = a[:, None] * nn + w[:, None] * k[t]
            den[t] = torch.maximum((nn * q[t]).sum(-1).abs(), torch.exp(-mm)) + 1e-6
            if whole:
                s = a[:, None, None] * s + (w[:, None] * k[t])[:, :, None] * v[t][:, None]
                num[t] = (q[t][:, None] @ s)[:, 0]
        if cnt:
            t += 1
            S[b], n[b], m[b] = s, nn, mm
    return num, den, S, n, m


@pytest.mark.parametrize("D,Dv", [(128, 72), (256, 136), (256, 64)])
def test_segments_mlstm(D, Dv):
    """Against float64, at the sizes whose normaliser is dealt to the waves once (128 rows) and twice (256): four segments."""
    from chronos.ops import hybrid as hops

    H, lens, starts = 2, [1100, 0, 513], [0, 3, 9]
    _in_chunks("mlstm", lens, H, D, Dv)
    T, B, g = sum(lens), len(lens), torch.Generator(device=DEV).manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    proj, gp = rnd(T, 2 * H * D + 2 * H * Dv).bfloat16(), rnd(T, 2 * H)
    gp[:, H:] += 3.0
    S0, n0, m0 = rnd(B, H, D, Dv) * 0.3, rnd(B, H, D) * 0.5, rnd(B, H)
    S, n, m = S0.clone(), n0.clone(), m0.clone()
    ranges = [torch.tensor(x, dtype=torch.int32, device=DEV) for x in ([0, 1100, 1100, T], starts, [0, 1, 2])]
    o = hops.mlstm_scan(proj, gp, *ranges, S, n, m, H, D, Dv, 9.0, max(lens))
    num, den, Sw, nw, mw = _mlstm(proj, gp, S0, n0, m0, lens, starts, 9.0)
    assert _rel(o * den[..., None], num) < 1e-5
    assert _rel(S, Sw) < 2e-6 and _rel(n, nw) < 2e-6 and _rel(m, mw) < 1e-6


@pytest.mark.parametrize("HK,H,D,Dv,form", [(1, 2, 128, 72, "token"), (2, 2, 128, 128, "head"), (1, 3, 256, 64, "token"), (2, 4, 64, 40, "token"),
                                            (1, 2, 128, 72, "rows"), (1, 2, 256, 64, "rows")])
def test_segments_scaled(HK, H, D, Dv, form):
    """Against float64: heads that share queries and keys, factors on queries, keys and values, with segments."""
    from chronos.ops import hybrid as hops

    lens, starts = [1100, 0, 513], [0, 3, 9]
    _in_chunks(form, lens, H, D, Dv)
    T, B, g = sum(lens), len(lens), torch.Generator(device=DEV).manual_seed(H * D + Dv)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    rand = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    proj = rnd(T, 2 * HK * D + H * Dv + 16).bfloat16()
    dec = 1 - rand(H) ** 4 if form == "head" else rand(T, H, D) ** (1 / 16) if form == "rows" else torch.exp(-0.2 * rand(T, H))
    if form == "token":
        dec[7::90], dec[11::400] = -0.9, 1.2
    qsc, ksc, vs = rand(T, HK), rand(T, HK), None if form == "head" else rand(T, H)
    S0 = rnd(B, H, D, Dv) * 0.3
    S = S0.clone()
    ranges = [torch.tensor(x, dtype=torch.int32, device=DEV) for x in ([0, 1100, 1100, T], starts, [0, 1, 2])]
    o = hops.linear_scan(proj, 8, 8 + HK * D, 8 + 2 * HK * D, qsc, ksc, 1.0, dec, None, *ranges, S, HK, H, D, Dv, vs, max(lens))
    p, rep = proj.double(), H // HK
    q = (p[:, 8:8 + HK * D].view(T, HK, D) * qsc.double()[..., None]).repeat_interleave(rep, 1)
    k = (p[:, 8 + HK * D:8 + 2 * HK * D].view(T, HK, D) * ksc.double()[..., None]).repeat_interleave(rep, 1)
    v = p[:, 8 + 2 * HK * D:8 + 2 * HK * D + H * Dv].view(T, H, Dv) * (vs.double()[..., None] if vs is not None else 1.0)
    d = (dec.double().expand(T, H) if dec.dim() < 3 else dec.double()).reshape(T, H, -1, 1)
    want, Sw, t = torch.empty(T, H, Dv, dtype=torch.double, device=DEV), S0.double(), 0
    for b, cnt in enumerate(lens):
        s = Sw[b] * float(starts[b] > 0)
        for t in range(t, t + cnt):
            s = d[t] * s + k[t][:, :, None] * v[t][:, None]
            want[t] = (q[t][:, None] @ s)[:, 0]
        if cnt:
            t, Sw[b] = t + 1, s
    assert _rel(o, want) < 2e-6 and _rel(S, Sw) < 2e-6
