"""The counters by which a split product's workgroups find their last one: zero for every graph, also when the first graph captured on a stream is
never replayed."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# few counters, of the buffers that are there; more of them (66048 tiles) than those hold, made in the capture
@pytest.mark.parametrize("m,n,k,mode,plan", [(30, 4096, 4096, 2, (74, 4)), (4096, 33024, 256, 0, (72, 2))])
def test_first_graph_never_replayed(m, n, k, mode, plan):
    from chronos import ops
    from chronos.ops import gemm as G

    ops.load()
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w = torch.randn(m, k, device="cuda", generator=g).bfloat16(), (torch.randn(n, k, device="cuda", generator=g) / 64).bfloat16()
    res = torch.zeros(m, n, device="cuda", dtype=torch.bfloat16) if mode == G.PP_RESID else None
    product = lambda: G.pp_gemm(x, w, mode, plan, resid=res)[0]  # noqa: E731
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
