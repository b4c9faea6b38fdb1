"""Queries and keys turned in pieces of 8 columns (csrc/hybrid/sandwich.hip rotate_qk_vec_kernel) against the general kernel, which rows off 16 bytes take, and
the plain reference."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# part and all of a head turned, none; one head, more pieces than threads; no keys' heads, no queries'
@pytest.mark.parametrize("HQ,HK,D,dims", [(1, 1, 16, 16), (8, 8, 128, 128), (8, 2, 128, 64), (32, 32, 128, 128), (3, 5, 64, 0), (2, 0, 24, 16), (0, 3, 40, 32)])
@pytest.mark.parametrize("T", [1, 37])
def test_pieces(HQ, HK, D, dims, T):
    from chronos.models.hybrid import rope_cos_sin
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    hops.load()
    g = torch.Generator(device=DEV).manual_seed(HQ * D + dims)
    n, q_off, k_off = (HQ + HK) * D + 24, 8, 16 + HQ * D
    proj = torch.randn(T, n, device=DEV, generator=g).bfloat16()
    pos = torch.tensor([(7 * t) % 60 for t in range(T)], dtype=torch.int32, device=DEV)
    tab = rope_cos_sin(1e4, dims, 64, DEV) if dims else None
    a, b, c = proj.clone(), torch.zeros(T, n + 1, device=DEV, dtype=torch.bfloat16), proj.clone()
    b[:, 1:] = proj
    hops.rotate_qk(a, q_off, k_off, HQ, HK, D, dims, tab, pos, 1.0, D ** -0.5)
    hops.rotate_qk(b, q_off + 1, k_off + 1, HQ, HK, D, dims, tab, pos, 1.0, D ** -0.5)
    ref.rotate_qk(c, q_off, k_off, HQ, HK, D, dims, tab, pos, 1.0, D ** -0.5)
    # one float32 sum of two products each (fused or not), rounded once: a last place of bfloat16 apart at most, of the larger term where they cancel
    big = proj.float().abs().max()
    for want in (b[:, 1:], c):
        assert float(((a.float() - want.float()).abs() - 2.0 ** -7 * want.float().abs()).max()) <= 2.0 ** -20 * float(big)
    assert torch.equal(a[:, :8], proj[:, :8]) and torch.equal(a[:, -8:], proj[:, -8:])
