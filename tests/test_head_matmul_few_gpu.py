"""Per-head products of few tokens: tokens around a workgroup's, columns and K off its tiles, gate columns, rows that are parts of wider ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 15, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("N,K", [(128, 512), (40, 256), (33, 264), (512, 128), (16, 8), (96, 520), (128, 1032)])
def test_few_tokens(T, N, K):
    from chronos.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    H = 3
    a, w = rnd(T, H, K + 8).bfloat16(), (rnd(H, N, K) * K ** -0.5).bfloat16()
    wide, src = rnd(T, H, N + 4).bfloat16(), rnd(T, 24 + H * N).bfloat16()
    keep = wide[:, :, N:].clone()
    want = torch.matmul(a[:, :, :K].double().transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()).transpose(0, 1)
    hops.head_matmul(a[:, :, :K], w, wide[:, :, :N])
    gated = hops.head_matmul(a[:, :, :K], w, None, src, 24)
    # float32 sums, rounded to bfloat16 once: 2^-9 of each value at most
    for got, ref in ((wide[:, :, :N], want), (gated, want * torch.sigmoid(src[:, 24:].double()).view(T, H, N))):
        assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all()
    assert torch.equal(wide[:, :, N:], keep)
