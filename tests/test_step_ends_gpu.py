"""The two ends of a hybrid decoder's step: first positions beside the embedding, norms of chosen rows, float32 logits."""
import pytest
import torch

from chronos.ops import gemm, hybrid as hops, hybrid_ref as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(*s, seed=0):
    return torch.randn(*s, generator=torch.Generator().manual_seed(seed)).to(DEV)


@pytest.mark.parametrize("lens", [[1], [5, 0, 7], [300, 1, 0], [0, 3]])
@pytest.mark.parametrize("dt,d", [(torch.bfloat16, 64), (torch.bfloat16, 60), (torch.float32, 36)])
def test_first_positions(lens, dt, d):
    qs = torch.tensor([0] + lens).cumsum(0).int().to(DEV)
    T = sum(lens)
    pos = torch.randint(0, 9999, (T,), generator=torch.Generator().manual_seed(1)).int().to(DEV)
    ids = torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(2)).int().to(DEV)
    table = _rand(50, d).to(dt)
    for emit in (True, False):
        x, h, p0 = hops.embed_start(ids, table, dt, 2.5, emit, pos, qs)
        wx, wh = ref.embed_rows(ids, table, dt, 2.5, emit)
        assert torch.equal(x, wx) and (h is None) == (wh is None) and (h is None or torch.equal(h, wh))
        assert torch.equal(p0, pos[qs[:-1].long().clamp(max=T - 1)])


def test_first_positions_of_other_layouts():
    """Positions that only the first of a sequence are taken of may lie in any stride and type, as the sequences' starts may."""
    qs = torch.tensor([0, 3, 7], device=DEV)
    pos = torch.arange(100, 114, dtype=torch.int32, device=DEV)[::2]
    ids, table = torch.arange(7, dtype=torch.int32, device=DEV), _rand(50, 64).bfloat16()
    for p, q in ((pos, qs.int()), (pos.long(), qs.int()), (pos.contiguous(), qs), (pos, qs)):
        x, h, p0 = hops.embed_start(ids, table, torch.bfloat16, 1.0, True, p, q)
        wx, wh = ref.embed_rows(ids, table, torch.bfloat16, 1.0, True)
        assert torch.equal(x, wx) and torch.equal(h, wh) and p0.dtype == p.dtype and p0.tolist() == [100, 106]


@pytest.mark.parametrize("d", [64, 1024, 1028, 4096, 4100, 30])
@pytest.mark.parametrize("idx", [[3], [0, 8, 8, 2, 5], []])
def test_chosen_rows(d, idx):
    x, w = _rand(9, d), _rand(d, seed=1)
    rows = torch.tensor(idx, dtype=torch.int64, device=DEV)
    for r in (rows, rows.int()):
        for at in (torch.bfloat16, torch.float32):
            forms = [lambda a, **k: hops.layer_norm(a, w, 1e-5, at, **k), lambda a, **k: hops.rms_norm(a, w, 1e-5, at, **k)]
            if d % 2 == 0:
                forms.append(lambda a, **k: hops.rms_norm(a, w, 1e-5, at, 2, **k))
            for f in forms:
                assert torch.equal(f(x, rows=r), f(x.index_select(0, r)))


def test_row_that_is_not_there():
    for d in (1024, 4096):
        x, w = _rand(4, d), _rand(d, seed=1)
        rows = torch.tensor([1, 4, -1], device=DEV)
        for y in (hops.layer_norm(x, w, 1e-5, torch.float32, rows), hops.rms_norm(x, w, 1e-5, torch.float32, 1, rows),
                  hops.rms_norm(x, w, 1e-5, torch.float32, 2, rows)):
            assert torch.isfinite(y[0]).all() and torch.isnan(y[1:]).all()


# (2048 x 512: 16-row tiles; 4096 x 11008: K split, its slices summed; 32768 x 1024: no split; 96 rows: the rounded product's values)
@pytest.mark.parametrize("m", [1, 2, 16, 17, 33, 64, 96])
@pytest.mark.parametrize("n,k", [(2048, 512), (32768, 1024), (4096, 11008), (4112, 4160)])
def test_float32_products(m, n, k):
    x, w = _rand(m, k).bfloat16(), (_rand(n, k, seed=1) * k ** -0.5).bfloat16()
    y = hops.matmul_f32(x, w)
    want = x.double() @ w.double().t()
    assert y.dtype == torch.float32 and y.shape == (m, n)
    own = gemm.product_f32(x, w) is not None
    # products of bfloat16 are exact in float32; k sums round to 2^-24 of partial sums of at most about 2 sqrt(k) of the result's size each
    off = (y.double() - want).norm() / want.norm()
    assert off < (k ** 0.5 * 2 ** -23 if own else 2 ** -8)
    assert own or m in (1, 33, 64, 96)


# a vocabulary's rows: whichever tiles the rules pick for up to 64 of them, the sums come unrounded
@pytest.mark.parametrize("m", [2, 32, 33, 48, 64])
@pytest.mark.parametrize("n,k", [(32768, 1024), (32768, 4096), (12288, 2048), (22016, 2816), (16388, 512)])
def test_float32_logits_of_any_rows(m, n, k):
    x, w = _rand(m, k).bfloat16(), (_rand(n, k, seed=1) * k ** -0.5).bfloat16()
    y = gemm.product_f32(x, w)
    if n % 16:   # (no rule takes it)
        assert y is None
        assert torch.equal(hops.matmul_f32(x, w), hops.matmul(x, w).float())
    else:
        want = x.double() @ w.double().t()
        assert (y.double() - want).norm() / want.norm() < k ** 0.5 * 2 ** -23
