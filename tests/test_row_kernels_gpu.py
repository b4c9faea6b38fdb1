"""The 16-bytes-per-lane forms of the row kernels (csrc/hybrid) at the sizes where they start, end and fall back, against the
PyTorch references.  Outputs are bfloat16 (2^-8 of the value between neighbours; the largest value's rounding plus that of a
float32 sum in another order: 1.2e-2 of the largest magnitude at most, as in the other kernel tests) or float32 (2e-5)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _g(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rand(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, device=DEV, generator=g) * scale).to(dtype)


def _close(a, b, tol):
    a, b = a.float(), b.float()
    assert float((a - b).abs().max()) <= tol * (float(b.abs().max()) + 1e-6)


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("rows", [1, 5, 64])
@pytest.mark.parametrize("d", [8, 520, 1024, 1032, 2048, 2056, 4096, 8192, 8200, 100])
def test_add_layer_norm(rows, d):
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    g = _g(rows + d)
    y, x, w = _rand(g, rows, d, dtype=BF, scale=3.0), _rand(g, rows, d), _rand(g, d)
    x2 = x.clone()
    h, h2 = hops.add_layer_norm(y, x, w, 1e-5, BF), ref.add_layer_norm(y, x2, w, 1e-5, BF)
    _close(x, x2, 2e-5)
    _close(h, h2, 1.2e-2)


@pytest.mark.parametrize("n", [8, 2048, 2056, 4100, 7])
@pytest.mark.parametrize("kind", [0, 1])
def test_act(n, kind):
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    x = _rand(_g(n), 3, n, dtype=BF, scale=3.0)
    x[0, 0], x[-1, -1] = 50.0, -50.0
    _close(hops.act_inplace(x.clone(), kind), ref.act_inplace(x.clone(), kind), 1.2e-2)


@pytest.mark.parametrize("H,Dv,off", [(3, 32, 8), (2, 64, 0), (5, 128, 16), (2, 256, 8), (1, 512, 8), (2, 96, 8), (3, 128, 3)])
@pytest.mark.parametrize("silu", [True, False])
def test_head_norm_gate(H, Dv, off, silu):
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    g = _g(H * Dv + off)
    o, src, w = _rand(g, 13, H, Dv), _rand(g, 13, off + H * Dv + 8, dtype=BF, scale=4.0), _rand(g, H * Dv)
    src[0, off], src[1, off] = 200.0, -200.0
    _close(hops.head_norm_gate(o, src, off, w, 1e-6, silu, BF), ref.head_norm_gate(o, src, off, w, 1e-6, silu, BF), 1.2e-2)


@pytest.mark.parametrize("C,K,off", [(8, 2, 0), (264, 3, 8), (2056, 4, 16), (4096, 4, 8), (64, 5, 8), (64, 4, 4)])
@pytest.mark.parametrize("many", [False, True])
def test_short_conv(C, K, off, many):
    """``many``: enough tokens for eight per thread; ranges start and end inside and on the edges of those blocks."""
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    lens = [2, 1, 8, 0, 1, 13, 3, 700, 1400, 8] if many else [1, 3, 0, 9]
    g = _g(C + K)
    starts = [(0, 5, 2, 7, 1, 0, 3, 9, 0, 4)[i] for i in range(len(lens))]
    slots = list(range(len(lens)))[::-1]
    qs = [0]
    for n in lens:
        qs.append(qs[-1] + n)
    seq = _i32([b for b, n in enumerate(lens) for _ in range(n)])
    x, w, bias = _rand(g, qs[-1], C + off + 8, dtype=BF), _rand(g, C, K, scale=0.5), _rand(g, C)
    hist = _rand(g, len(lens) + 1, K - 1, C, dtype=BF)
    hist2 = hist.clone()
    for b, silu in ((bias, True), (None, False)):
        y = hops.short_conv(x, w, seq, _i32(qs), _i32(starts), _i32(slots), hist, silu, b, off)
        y2 = ref.short_conv(x, w, _i32(qs), _i32(starts), _i32(slots), hist2, silu, b, off)
        _close(y, y2, 8e-3)
        assert torch.equal(hist, hist2)


def test_short_conv_of_many_tokens():
    """More blocks of eight tokens than a second grid axis holds."""
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    C, K, lens = 8, 3, [8 * 65535 + 1, 20]
    T, g = sum(lens), _g(1)
    x, w = _rand(g, T, C, dtype=BF), _rand(g, C, K)
    seq = torch.arange(2, device=DEV, dtype=torch.int32).repeat_interleave(torch.tensor(lens, device=DEV))
    qs, zero, slots, hist = _i32([0, lens[0], T]), _i32([0, 0]), _i32([0, 1]), torch.zeros(2, K - 1, C, device=DEV, dtype=BF)
    y = hops.short_conv(x, w, seq, qs, zero, slots, hist.clone(), True, None, 0)
    _close(y, ref.short_conv(x, w, qs, zero, slots, hist.clone(), True, None, 0), 8e-3)


@pytest.mark.parametrize("H,G,D,Dv,dims,norm,v_rot,v_k", [
    (8, 2, 128, 128, 64, True, False, False), (4, 1, 64, 64, 64, True, True, False), (3, 3, 128, 128, 16, False, False, True),
    (2, 1, 256, 64, 0, False, False, False), (2, 2, 512, 32, 256, True, True, False), (4, 2, 8, 8, 0, True, False, False),
    (6, 2, 32, 48, 32, True, True, False), (2, 1, 128, 128, 8, True, False, False), (2, 1, 96, 96, 32, True, False, False)])
@pytest.mark.parametrize("mix", [False, True])
def test_window_prep(H, G, D, Dv, dims, norm, v_rot, v_k, mix):
    from chronos.models.hybrid import rope_cos_sin
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    g = _g(H * D + Dv + dims)
    T, NB, bs = 9, 7, 16
    off = H * D if v_k else -1
    width = max((H + G) * D + G * Dv, 0) + 8
    qkv = _rand(g, T, width, dtype=BF)
    pos, seq = _i32([0, 1, 2, 30, 31, 32, 5, 6, 47]), _i32([0, 0, 0, 1, 1, 1, 2, 2, 1])
    bt = _i32([[1, 0, 0], [2, 3, 4], [5, 6, 0]])
    kc, vc = _rand(g, NB, bs, G, D, dtype=BF), _rand(g, NB, bs, G, Dv, dtype=BF)
    kc2, vc2 = kc.clone(), vc.clone()
    qn, kn = (_rand(g, D) + 1, _rand(g, D) + 1) if norm else (None, None)
    vf, lam = (_rand(g, T, G * Dv, dtype=BF), _rand(g, 1)) if mix else (None, None)
    cs = rope_cos_sin(1e4, dims, 64, DEV) if dims else None
    vcs = rope_cos_sin(1e4, Dv, 64, DEV) if v_rot else None
    temp = torch.rand(64, device=DEV, generator=g) if mix else None
    a, b = qkv.clone(), qkv.clone()
    v1 = hops.window_prep(a, H, G, D, Dv, vf, lam, pos, seq, bt, qn, kn, 1e-6, cs, dims, kc, vc, not mix, off, vcs, temp)
    v2 = ref.window_prep(b, H, G, D, Dv, vf, lam, pos, seq, bt, qn, kn, 1e-6, cs, dims, kc2, vc2, not mix, off, vcs, temp)
    for x, y in ((a, b), (kc, kc2), (vc, vc2)):
        _close(x, y, 1.2e-2)
    assert torch.equal(a[:, H * D:], qkv[:, H * D:]), "only queries are rewritten"
    if not mix:
        assert torch.equal(v1, v2)


@pytest.mark.parametrize("T,F,pad", [(1, 8, 0), (3, 2056, 0), (5, 2064, 8), (4, 12, 0), (2, 2048, 4)])
def test_glu(T, F, pad):
    """16 bytes per lane and what does not allow it (F % 8, rows off 16 bytes).  Tolerance: the result's rounding to bfloat16, half a last
    place or 2^-8 of the value, and the hardware's sigmoid, 1e-6."""
    from chronos.ops import hybrid as hops

    g = torch.Generator(device=DEV).manual_seed(F)
    gu = (torch.randn(T, 2 * F + pad, device=DEV, generator=g) * 4).bfloat16()
    y = torch.empty(T, F + pad, device=DEV, dtype=torch.bfloat16)
    hops.glu_cols(gu, 0, F, 7.0, 1.702, 1.0, y[:, :F])
    a, u = gu[:, :F].double().clamp(max=7.0), gu[:, F:2 * F].double().clamp(-7.0, 7.0)
    want = a * torch.sigmoid(1.702 * a) * (u + 1.0)
    assert ((y[:, :F].double() - want).abs() <= want.abs() * (2 ** -8 + 1e-5) + 1e-6).all()


@pytest.mark.parametrize("n,p", [(4, 1 / 16), (4099, 1 / 16), (4096, 1 / 8), (4096, 1.0), (4096, 2.5)])
def test_decay_pow(n, p):
    """Both forms, at the ends of the range: a few float32 roundings of p log sigmoid(z) (2^-24 of up to 7 p) and of the result."""
    from chronos.ops import hybrid as hops

    g = torch.Generator(device=DEV).manual_seed(n)
    z = torch.randn(n, device=DEV, generator=g) * 4
    z[:4] = torch.tensor([float("inf"), -float("inf"), 100.0, 0.0], device=DEV)
    want = torch.exp(p * torch.nn.functional.logsigmoid(z.double()))
    got = hops.decay_pow(z.clone(), p)
    assert ((got.double() - want).abs() <= want * (2 ** -22 + 2 ** -20 * p)).all()
    nan = torch.full((4,), float("nan"), device=DEV)
    assert hops.decay_pow(nan, p).isnan().all()


def test_gated_unit_sigmoid():
    """a sigmoid(slope a), every bfloat16 a from -60 to 30 and 150 slopes, against float64.  A float32 result off by n units of its last
    place rounds to another bfloat16 than the exact one in n / 32768 of the cases at most (bfloat16 keeps 16 bits less): with the 4 units
    that the sigmoid and two products may be off, 1.3e-4 of them.  No result is further off than the rounding to bfloat16 (2^-8), where the
    sigmoid is below float32's normal numbers neither (slope a down to -88.2)."""
    from chronos.ops import hybrid as hops

    a = torch.arange(-32768, 32768, dtype=torch.int32, device=DEV).to(torch.int16).view(BF)
    a = a[(a >= -60) & (a <= 30) & (a.abs() > 2 ** -10)]
    a = a[:a.numel() // 8 * 8].view(1, -1)
    gu, wrong, total = torch.cat([a, torch.zeros_like(a)], 1), 0, 0
    for i in range(150):
        slope = float(torch.tensor(0.5 + 0.97 * i / 149, dtype=torch.float32))
        z = (a.float() * slope).double()
        y, want = hops.glu(gu, 1e30, slope, 1.0, BF), (a.double() * torch.sigmoid(z))
        wrong += int((y != want.to(BF)).sum())
        total += a.numel()
        assert float(((y.double() - want).abs() - want.abs() * 2 ** -7.9).max()) <= 0
    assert total > 400_000 and wrong <= 1.3e-4 * total, (wrong, total)


@pytest.mark.parametrize("tau", [16.0, 20.0, 64.0])
@pytest.mark.parametrize("lo,hi", [(-100.0, -20.0), (-20.0, -4.0), (-4.0, 4.0), (4.0, 60.0)])
def test_decay_pow_error(tau, lo, hi):
    """Relative error of sigmoid(z)^(1 / tau) as a float32.  The logarithm and its product with 1 / tau round once each, 2^-24 of at most
    100 / tau, which the exponential turns into a relative error; the exponential itself and the result: 2 units, 2^-23."""
    from chronos.ops import hybrid as hops

    z = (torch.rand(1 << 16, device=DEV, generator=_g(int(tau))) * (hi - lo) + lo).view(16, -1)
    p = float(torch.tensor(1 / tau, dtype=torch.float32))
    want = torch.exp(torch.nn.functional.logsigmoid(z.double()) * p)
    rel = ((hops.decay_pow(z.clone(), p).double() - want) / want).abs().max()
    size = max(-lo, 0.7) / tau
    assert float(rel) <= 2 ** -23 + (0 if tau in (16.0, 64.0) and hi <= -4 else size * 2 ** -23)
