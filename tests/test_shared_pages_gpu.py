"""Decode attention over pages that rows share (csrc/kernels/attention.hip neighbour_pages): a row's output depends on what its pages hold,
not on who else holds them, so tables whose rows share leading pages give the bits of tables whose every row has copies of its own."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BS, D, HKV, HQ = "cuda", 16, 128, 8, 32


def _tables(ctx, shared):
    """(table of rows that share, table of rows with copies, page of the first -> page of the second).  shared[b]: leading pages that row b
    has in common with every other row; the rest, and always the last, is its own."""
    nbs = [-(-c // BS) for c in ctx]
    width, common, at = max(nbs) + 3, max(shared), 1 + max(shared)
    one, two = torch.zeros(len(ctx), width, dtype=torch.int32), torch.zeros(len(ctx), width, dtype=torch.int32)
    src, free = [], 1
    for b, n in enumerate(nbs):
        s = min(shared[b], n - 1)
        row = list(range(1, 1 + s)) + list(range(at, at + n - s))
        at += n - s
        one[b, :n], two[b, :n] = torch.tensor(row, dtype=torch.int32), torch.arange(free, free + n, dtype=torch.int32)
        src += row
        free += n
    return one.to(DEV), two.to(DEV), at, torch.tensor([0] + src, device=DEV)


def _pages(n, fp8, seed):
    from chronos.ops import reference as ref

    g = torch.Generator(device=DEV).manual_seed(seed)
    k, v = torch.randn(n, HKV, BS, D, device=DEV, generator=g), torch.randn(n, HKV, D, BS, device=DEV, generator=g)
    return (ref.to_fp8_bytes(k, 2.0), ref.to_fp8_bytes(v, 4.0)) if fp8 else (k.to(torch.bfloat16), v.to(torch.bfloat16))


ROWS = 130   # with 8 heads more than the 1024 items from which one wave takes a row
MIXES = {"all of one template": lambda b, n: 5, "to the last page": lambda b, n: n, "none": lambda b, n: 0,
         "every other row": lambda b, n: 6 if b % 2 else 0, "the second half": lambda b, n: 7 if b >= 65 else 0,
         "beyond a window of 64": lambda b, n: 70}


@pytest.mark.parametrize("mix", sorted(MIXES))
def test_one_wave_a_row(mix):
    from chronos import ops
    from chronos.models.llama import get_config, rope_table
    from chronos.ops import reference as ref

    g = torch.Generator().manual_seed(7)
    ctx = torch.randint(1, 260, (ROWS,), generator=g).tolist()
    ctx[:10] = [1, 16, 17, 32, 33, 1008, 1040, 1041, 1300, 1290]
    one, two, pages, src = _tables(ctx, [MIXES[mix](b, -(-c // BS)) for b, c in enumerate(ctx)])
    k1, v1 = _pages(pages, False, 3)
    k2, v2 = k1[src].contiguous(), v1[src].contiguous()
    cl, qs = torch.tensor(ctx, dtype=torch.int32, device=DEV), torch.arange(ROWS + 1, dtype=torch.int32, device=DEV)
    gd = torch.Generator(device=DEV).manual_seed(5)
    qkv = torch.randn(ROWS, (HQ + 2 * HKV) * D, device=DEV, generator=gd).to(torch.bfloat16)
    q = qkv.view(ROWS, -1, D)[:, :HQ].contiguous()
    plain = [ops.paged_attention(q, k, v, bt, qs, cl, None, ROWS, 1, 1) for k, v, bt in ((k1, v1, one), (k2, v2, two))]
    assert torch.equal(*plain)
    want = ref.paged_attention(q, k1, v1, one, qs, cl, None, ROWS, 1, 1)
    assert float((plain[0].float() - want.float()).norm() / want.float().norm()) < 1e-2   # (probabilities and outputs of 8 bits: 2^-8)
    cs = rope_table(get_config("llama3.1-8b"), 2048, DEV)
    fused = [ops.decode_attention_rope(qkv, cl - 1, cs, k, v, bt, cl, ROWS, HQ, 1 / math.sqrt(D)) for k, v, bt in ((k1, v1, one), (k2, v2, two))]
    assert torch.equal(*fused)
    last = [bt.gather(1, ((cl - 1) // BS).long()[:, None])[:, 0].long() for bt in (one, two)]
    assert torch.equal(k1[last[0]], k2[last[1]]) and torch.equal(v1[last[0]], v2[last[1]])   # the new tokens' pages


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("ctx,share,nsplit", [([700], 0, 4), ([700, 690], 20, 3), ([2000, 1990, 33, 1, 1500], 60, 4), ([5000, 4990, 40], 1000, 16),
                                              ([513, 512, 511, 1026], 32, 2)])
def test_split_over_workgroups(ctx, share, nsplit, fp8):
    from chronos import ops
    from chronos.ops import reference as ref

    one, two, pages, src = _tables(ctx, [share] * len(ctx))
    k1, v1 = _pages(pages, fp8, len(ctx))
    k2, v2 = k1[src].contiguous(), v1[src].contiguous()
    n, scales = len(ctx), (0.5, 0.25) if fp8 else (1.0, 1.0)
    cl, qs = torch.tensor(ctx, dtype=torch.int32, device=DEV), torch.arange(n + 1, dtype=torch.int32, device=DEV)
    q = torch.randn(n, HQ, D, device=DEV, generator=torch.Generator(device=DEV).manual_seed(9)).to(torch.bfloat16)
    got = [ops.paged_attention(q, k, v, bt, qs, cl, None, n, 1, nsplit, None, *scales) for k, v, bt in ((k1, v1, one), (k2, v2, two))]
    assert torch.equal(*got)
    want = ref.paged_attention(q, k1, v1, one, qs, cl, None, n, 1, 1, None, *scales)
    assert float((got[0].float() - want.float()).norm() / want.float().norm()) < 1e-2
