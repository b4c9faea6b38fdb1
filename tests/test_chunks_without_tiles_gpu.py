"""The recurrences' chunks that make their tiles on their way (csrc/hybrid/gla_scan.hip gla_scan_kernel, chunk_scan.hip with the delta rule), which calls take whose tiles
would need more scratch than they may have: the tests of the chunks, segments and values that are not finite, with no scratch for tiles."""
import functools

import pytest
import torch

import test_chunk_scan_gpu as chunks
import test_not_finite_gpu as not_finite

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_tiles(monkeypatch):
    from chronos.ops import hybrid as hops

    monkeypatch.setattr(hops, "linear_scan", functools.partial(hops.linear_scan, tiles_mb=0))


@pytest.mark.parametrize("sizes", [(2, 4, 32, 40, True), (1, 2, 64, 64, False), (3, 3, 128, 72, True), (2, 2, 256, 128, False)])
def test_rows(sizes):
    chunks.test_rows(*sizes)


@pytest.mark.parametrize("lens,starts", [([1100, 40, 0, 513, 1023], [0, 3, 5, 9, 0]), ([2500], [7])])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
def test_segments(lens, starts, D):
    chunks.test_segments(lens, starts, "rows", D)


@pytest.mark.parametrize("sizes", [(1, 2, 128, 72), (1, 2, 256, 64)])
def test_segments_scaled(sizes):
    chunks.test_segments_scaled(*sizes, "rows")


@pytest.mark.parametrize("what,at,value", not_finite.WHERE)
@pytest.mark.parametrize("form", ["rows", "delta"])
def test_where_they_appear(form, what, at, value):
    not_finite.test_where_they_appear(form, what, at, value)


@pytest.mark.parametrize("D,Dv", [(32, 40), (128, 64), (256, 64)])
@pytest.mark.parametrize("form", ["rows", "delta"])
def test_sizes(form, D, Dv):
    not_finite.test_sizes(form, D, Dv)


@pytest.mark.parametrize("what,at,value", [("v", 5, not_finite.INF), ("v", 400, not_finite.NAN), ("k", 640, not_finite.INF), ("q", 300, not_finite.INF), ("decay", 200, not_finite.NAN),
                                           ("S", 0, not_finite.INF)])
def test_segments_not_finite(what, at, value):
    not_finite.test_segments("rows", what, at, value)


def test_which_form(monkeypatch):
    """Without scratch the other form does run: the delta rule's bits are the same, gated linear attention's read-outs differ in their last."""
    from chronos.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(1)
    T, H, D, Dv = 700, 2, 128, 64
    y, S0 = torch.randn(T, H * (2 * D + Dv), device="cuda", generator=g).bfloat16(), torch.randn(1, H, D, Dv, device="cuda", generator=g)
    decay = torch.rand(T, H, D, device="cuda", generator=g) ** 0.1
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    got = [hops.linear_scan(y, 0, H * D, 2 * H * D, None, None, 1.0, decay, None, i32([0, T]), i32([1]), i32([0]), S0.clone(), H, H, D, Dv, None, T, **mb)
           for mb in ({}, dict(tiles_mb=0), dict(tiles_mb=512))]
    assert torch.equal(got[0], got[1]) and not torch.equal(got[0], got[2])
