"""The counters by which a split product's workgroups find their last one: zero for every graph, also when the first graph captured on a stream is
never replayed."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_first_graph_never_replayed():
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w = torch.randn(30, 4096, device="cuda", generator=g).bfloat16(), (torch.randn(4096, 4096, device="cuda", generator=g) / 64).bfloat16()
    res = torch.zeros(30, 4096, device="cuda", dtype=torch.bfloat16)
    product = lambda: G.pp_gemm(x, w, G.PP_RESID, (74, 4), resid=res)[0]  # noqa: E731
    want = product()
    stream, pool = torch.cuda.Stream(), torch.cuda.graph_pool_handle()
    dirty = torch.cuda.CUDAGraph()
    with torch.cuda.graph(dirty, pool=pool, stream=stream):   # what lies in the pool's memory
        junk = [torch.full((1 << 16,), 1 << 20, device="cuda", dtype=torch.int32) for _ in range(24)]
    dirty.replay()
    torch.cuda.synchronize()
    del junk
    first, second = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(first, pool=pool, stream=stream):
        y0 = product()
    with torch.cuda.graph(second, pool=pool, stream=stream):
        y = product()
    for _ in range(3):
        y.fill_(float("nan"))
        second.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    first.replay()
    torch.cuda.synchronize()
    assert torch.equal(y0, want)
