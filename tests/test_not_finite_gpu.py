"""Infinities and NaN in the recurrences' prompt kernels (csrc/hybrid/chunk_scan.hip, gla_scan.hip) against the plain recurrence of hybrid_ref
in float32: they appear where a token-by-token recurrence has them, as what it has, and never at tokens before the one that brings
them; everything else keeps its value (4e-6: both sides round, as in the other tests of these kernels)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
INF, NAN = float("inf"), float("nan")
# (what, token, value): tokens of the second sequence
WHERE = [("v", 5, INF), ("v", 63, NAN), ("v", 64, -INF), ("v", 99, INF), ("k", 5, INF), ("k", 70, NAN), ("q", 17, -INF), ("q", 66, NAN), ("decay", 7, NAN),
         ("decay", 80, INF), ("S", 0, INF), ("S", 0, NAN), ("S", 0, 3.4e38), ("v", 40, 3e38)]


def _same(got, want):
    got, want = got.cpu().double(), want.cpu().double()
    assert torch.equal(got.isnan(), want.isnan()), "NaN elsewhere"
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[got.isinf()], want[want.isinf()]), "infinities elsewhere"
    # by size: roundings are relative to the sums' terms, so the values around a very large one say nothing by themselves
    for part in (want.abs() < 1e30, want.isfinite() & (want.abs() >= 1e30)):
        if part.any():
            assert float((got[part] - want[part]).norm() / want[part].norm()) < 4e-6


def _run(form, H, HK, D, Dv, lens, what, at, value, starts=(0, 3), seed=0):
    from chronos.ops import hybrid as hops

    T, g = sum(lens), torch.Generator().manual_seed(seed + D + Dv)
    hops.load()
    assert torch.ops.chronos.hy_chunk_scan_pays({"mlstm": 1, "delta": 2, "rows": 3}.get(form, 0), T, len(lens), H, D, Dv, max(lens))   # in chunks
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    rand = lambda *s: torch.rand(*s, generator=g)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    t = lens[0] + at
    proj, S, n, m, gp = rnd(T, 2 * HK * D + H * Dv + 8).bfloat16(), rnd(3, H, D, Dv), rnd(3, H, D), rnd(3, H), rnd(T, 2 * H)
    if form.startswith("delta"):
        proj[:, HK * D:2 * HK * D] *= D ** -0.5   # (a stable recurrence: keys of unit length)
    decay = rand(H) * 0.2 + 0.8 if form == "fixed" else (rand(T, H, D) if form == "rows" else rand(T, H)) ** 0.1
    beta, vs = rand(T, H) if form == "delta" else None, rand(T, H) if form == "token" else None
    col = {"q": D // 3, "k": HK * D + D // 2, "v": 2 * HK * D + Dv // 2}
    if what in col:
        proj[t, col[what]] = value
    elif what == "S":
        S[1, H - 1, 2, 7] = value
    elif form == "mlstm":
        gp[t, H] = value
    elif form == "fixed":
        decay[0] = value
    else:
        decay[t] = value

    def run(dev, most=max(lens)):
        p, q, p0, sl, St = (x.to(dev, copy=True) for x in (proj, i32([0, lens[0], T]), i32(starts), i32([2, 1]), S))
        if form == "mlstm":
            st = [St, n.to(dev, copy=True), m.to(dev, copy=True)]
            return hops.mlstm_scan(p, gp.to(dev), q, p0, sl, *st, H, D, Dv, 9.0, most), *st
        to = lambda x: None if x is None else x.to(dev)  # noqa: E731
        return hops.linear_scan(p, 0, HK * D, 2 * HK * D, None, None, 0.3, to(decay), to(beta), q, p0, sl, St, HK, H, D, Dv, to(vs), most), St

    # A gate that is NaN leaves the running maximum alone in the kernels, and they scale a read-out after its sum, which may overflow before:
    # there against the token-by-token kernels, which launches of short ranges take.
    for a, b in zip(run(DEV), run(DEV, 2) if form == "mlstm" and what == "decay" or value == 3.4e38 else run("cpu")):
        _same(a, b)


@pytest.mark.parametrize("what,at,value", WHERE)
@pytest.mark.parametrize("form", ["fixed", "token", "rows", "delta", "mlstm"])
def test_where_they_appear(form, what, at, value):
    if what == "decay" and form == "mlstm" and value == INF:
        value = NAN   # (a gate is bounded: an infinite pre-activation is an ordinary one)
    _run(form, 2, 2 if form == "mlstm" else 1, 64, 72, [33, 100], what, at, value)


@pytest.mark.parametrize("D,Dv", [(32, 40), (128, 64), (256, 64)])
@pytest.mark.parametrize("form", ["token", "rows", "delta", "mlstm"])
def test_sizes(form, D, Dv):
    if form == "delta" and D == 256:
        D = 128
    for what, at, value in (("v", 70, INF), ("k", 20, NAN), ("S", 0, INF)):
        _run(form, 1, 1, D, Dv, [20, 90], what, at, value)


@pytest.mark.parametrize("what,at,value", [("v", 5, INF), ("v", 400, NAN), ("k", 640, INF), ("q", 300, INF), ("decay", 200, NAN), ("S", 0, INF)])
@pytest.mark.parametrize("form", ["fixed", "token", "rows", "mlstm"])
def test_segments(form, what, at, value):
    """One long sequence in segments side by side: what an early one brings reaches the later ones."""
    _run(form, 2, 2, 64, 64, [40, 700], what, at, value)
