"""Windowed attention's workgroup order and key splits (csrc/hybrid/window_attention_mfma.hip): launches of more than 512
workgroups (late blocks first), of fewer (the second half the other way round, odd and even block counts) and with the keys split,
against float32 attention.

Tolerance: the softmax weights enter as two bfloat16 terms, the result is rounded to bfloat16, at most 2^-9 of its norm on average over random
values; float32 sums add 1e-5.  Checked: norm of the difference below 2^-8 of the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,T,window,keep", [(20, 900, 0, 0), (9, 900, 100, 3), (3, 65, 0, 0), (5, 129, 64, 0), (1, 1500, 0, 0), (8, 300, 512, 4)])
def test_order(B, T, window, keep):
    from chronos.ops import hybrid as hops

    H, G, D, BS = 8, 2, 64, 16
    g = torch.Generator(device=DEV).manual_seed(B * T)
    qkv, per = torch.randn(B * T, (H + 2 * G) * D, device=DEV, generator=g).bfloat16(), (T + BS - 1) // BS
    kc, vc = (torch.randn(B * per + 1, BS, G, D, device=DEV, generator=g).bfloat16() for _ in range(2))
    bt = (1 + torch.randperm(B * per, device=DEV, generator=g)).int().view(B, per)
    o = hops.window_attention(qkv, kc, vc, bt, torch.arange(B + 1, device=DEV).int() * T, torch.arange(T, device=DEV).int().repeat(B),
                              None, None, D ** -0.5, window, keep, H, torch.bfloat16, T).view(B, T, H, D)
    i = torch.arange(T, device=DEV)
    hide = i[None] > i[:, None]
    if window:
        hide |= (i[None] <= i[:, None] - window) & (i[None] >= keep)
    for b in range(B):
        k, v = (c[bt[b].long()].reshape(-1, G, D)[:T].float().repeat_interleave(H // G, 1) for c in (kc, vc))
        q = qkv[b * T:(b + 1) * T, :H * D].float().view(T, H, D)
        s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0)) * D ** -0.5
        want = torch.matmul(torch.softmax(s.masked_fill_(hide, float("-inf")), -1), v.transpose(0, 1)).transpose(0, 1)
        assert float((o[b].float() - want).norm() / want.norm()) < 2 ** -8, b


@pytest.mark.parametrize("lens,past", [([900, 1, 65, 0, 1, 300], [0, 700, 0, 5, 40, 100]), ([130] + [1] * 9, [16] + [200] * 9),
                                       ([33, 700, 2] * 8, [0, 64, 300] * 8), ([17, 1, 1], [480, 1, 333])])
@pytest.mark.parametrize("window,keep", [(0, 0), (100, 3)])
def test_order_of_unequal_sequences(lens, past, window, keep):
    """Prompts beside decode rows: every sequence's blocks are its own number, in its own order, with and without splits of the keys."""
    from chronos.ops import hybrid as hops

    H, G, D, BS = 8, 2, 64, 16
    B, T, g = len(lens), sum(lens), torch.Generator(device=DEV).manual_seed(sum(lens))
    qkv, per = torch.randn(T, (H + 2 * G) * D, device=DEV, generator=g).bfloat16(), max((n + c + BS - 1) // BS for n, c in zip(lens, past))
    kc, vc = (torch.randn(B * per + 1, BS, G, D, device=DEV, generator=g).bfloat16() for _ in range(2))
    bt = (1 + torch.randperm(B * per, device=DEV, generator=g)).int().view(B, per)
    qs = [sum(lens[:b]) for b in range(B + 1)]
    pos = torch.cat([torch.arange(c, c + n) for n, c in zip(lens, past)]).int().to(DEV)
    o = hops.window_attention(qkv, kc, vc, bt, torch.tensor(qs).int().to(DEV), pos, None, None, D ** -0.5, window, keep, H, torch.bfloat16, max(lens)).view(T, H, D)
    for b, (n, c) in enumerate(zip(lens, past)):
        if n == 0:
            continue
        k, v = (x[bt[b].long()].reshape(-1, G, D)[:c + n].float().repeat_interleave(H // G, 1) for x in (kc, vc))
        q = qkv[qs[b]:qs[b + 1], :H * D].float().view(n, H, D)
        i, p = torch.arange(c + n, device=DEV)[None], torch.arange(c, c + n, device=DEV)[:, None]
        hide = i > p
        if window:
            hide = hide | ((i <= p - window) & (i >= keep))
        s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) * D ** -0.5
        want = torch.matmul(torch.softmax(s.masked_fill_(hide, float("-inf")), -1), v.transpose(0, 1).contiguous()).transpose(0, 1)
        assert float((o[qs[b]:qs[b + 1]].float() - want).norm() / want.norm()) < 2 ** -8, b
