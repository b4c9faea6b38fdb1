"""A post-norm join whose rows every workgroup of the product behind it makes itself (csrc/kernels/gemm_skinny.hip JoinRows), against the join and the
product as launches of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(m, k, n, S, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    y = rnd(S, m, k) if S else rnd(m, k).bfloat16()
    return y, rnd(m, k), 1 + 0.1 * rnd(k), (rnd(n, k) * k ** -0.5).bfloat16(), rnd(40)


# one wave's run of columns and all of them; several rows to a run of workgroup's threads; slices 1 to 8 and rows
@pytest.mark.parametrize("m,k", [(1, 256), (1, 1024), (1, 2048), (1, 4096), (2, 1024), (3, 512), (5, 768), (16, 256)])
@pytest.mark.parametrize("S", [0, 1, 3, 8])
def test_join_in_front(m, k, S):
    from chronos import ops
    from chronos.ops import hybrid as hops

    hops.load()
    op = ops._k()
    y, x, wn, w, bias = _inputs(m, k, 1120, S, m * k + S)
    x0, x1 = x.clone(), x.clone()
    h1 = hops.scale_add_rms_norm(y, x1, wn, 2.0, 1e-6, torch.bfloat16)
    for cfg, mode, n0, nf in ((14, 0, 0, 0), (15, 0, 0, 0), (14, 0, 1080, 40), (15, 0, 1080, 40), (15, 3, 0, 0)):
        h = torch.empty(m, k, device=DEV, dtype=torch.bfloat16)
        out, few, xn = op.gemm_join(y, x, wn, 2.0, 1e-6, h, w, cfg, mode, n0, nf, bias if nf else None, 7.0, 1.7, 1.0)
        assert torch.equal(x, x0)
        # the same float32 arithmetic, the sum of squares in another order of its 256-column parts
        assert float(((xn - x1).abs() / x1.abs().clamp_min(1e-3)).max()) < 1e-5
        assert torch.equal(h, xn.bfloat16()) and float((h != h1).float().mean()) < 0.01
        want, wfew = op.gemm_few(h, w, cfg, mode, n0, nf, bias if nf else None, 7.0, 1.7, 1.0) if nf or mode else (op.gemm_slices(h, w, cfg, 1, True)[0].bfloat16(), None)
        assert torch.equal(out, want) and (not nf or torch.equal(few, wfew))


def _decode_rows(model, rows, ctx, vocab):
    """A step of one token a row behind ctx cached ones, and pages that hold them."""
    from chronos import ops
    from chronos.models.llama import StepBatch

    per = ctx // 16 + 1
    i32 = dict(dtype=torch.int32, device=DEV)
    pos, ar = torch.full((rows,), ctx, **i32), torch.arange(rows + 1, **i32)
    ids = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(6)).int().to(DEV)
    sb = StepBatch(ids, pos, ar[:rows], torch.arange(1, 1 + rows * per, **i32).view(rows, per), ar, pos + 1, torch.arange(rows, device=DEV), None, rows, 1,
                   ops.pick_nsplit(rows * model.hkv, ctx + 1), slots=ar[:rows].clone(), max_q=1)
    cache, g = model.make_cache(1 + rows * per, 16, rows), torch.Generator(device=DEV).manual_seed(9)
    for name in ("S", "n", "m", "lat", "kc", "vc", "kp", "vp", "hist"):
        for t in getattr(cache, name).values():
            t.normal_(0.0, 0.5, generator=g)
    return sb, cache


@pytest.mark.parametrize("rows", [1, 2, 3])
def test_model_steps(rows, monkeypatch):
    """Decode steps of a design with all three readers, with the joins in their products and with every join a launch: the same to rounding."""
    from chronos import ops
    from chronos.models import kalesun
    from chronos.models.hybrid import HybridDecoder
    from chronos.ops import hybrid as hops
    from chronos.utils import design_bench as db

    ops.load()
    hops.load()
    ops.device_init()
    size = db.KALESUN_SIZES["1k"]
    design = db.kalesun_config(size)
    for layer in design["layers"]:   # (a router's choice may turn on a last bit)
        if layer["mlp"]["kind"] == "moe":
            layer["mlp"] = dict(kind="dense", ff=size["ff"], limit=7.0)
    cfg = kalesun.config_from_dict(design)
    model = HybridDecoder(cfg, kalesun.pack_weights(cfg, kalesun.random_tensors(cfg, 3), DEV, torch.bfloat16), torch.device(DEV, 0), 8192, torch.bfloat16)
    assert size["width"] == 1024
    got, taken = [], []
    product = hops.JoinedRows.product

    def counted(self, *a, **k):
        r = product(self, *a, **k)
        taken.append(r is not None)
        return r

    monkeypatch.setattr(hops.JoinedRows, "product", counted)
    for joined in (True, False):
        if not joined:
            monkeypatch.setattr(hops.JoinedRows, "serves", staticmethod(lambda y, x: False))
        sb, cache = _decode_rows(model, rows, 70, cfg.vocab_size)
        with torch.no_grad():
            got.append(model.forward(sb, cache).double())
    assert (sum(taken) == 7) == (rows <= 2) and (len(taken) == 0) == (rows > 2)   # eight joins, the last has no reader
    # bfloat16 activations whose last bits differ here and there
    assert float((got[0] - got[1]).norm() / got[1].norm()) < 0.01


def test_registered_kernel_gets_its_product():
    """A kernel registered for the product is called, whatever stands in front of it."""
    from chronos.ops import gemm
    from chronos.ops import hybrid as hops

    hops.load()
    y, x, wn, w, _ = _inputs(1, 1024, 1120, 2, 3)
    calls = []
    entry = (lambda m, n, k: (n, k) == (1080, 1024), lambda a, b: calls.append(tuple(b.shape)) or a @ b.t())
    gemm._custom.append(entry)
    try:
        joined = hops.JoinedRows(y, x, wn, 2.0, 1e-6)
        out, few = hops.matmul_rowdot(joined, w[:1080], w[1080:], None, (w, 1080, 40))
    finally:
        gemm._custom.remove(entry)
    assert calls == [(1080, 1024)] and out.shape == (1, 1080) and few.shape == (1, 40) and joined.stream() is x
