"""Windowed attention of decode rows whose key tiles are a workgroup each (csrc/hybrid/window_attention_mfma.hip hy_window_nsplit)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# lengths around a tile's edges, 3 and 4 tiles, 16 and 17, splits without a key; windows and kept tokens in other tiles
@pytest.mark.parametrize("lens", [[1], [64], [65], [130], [191], [192], [200], [640], [641, 3], [700, 64, 129], [960], [1023], [1024, 30], [1500]])
@pytest.mark.parametrize("window,keep", [(0, 0), (512, 4), (100, 70)])
def test_decode_rows(lens, window, keep):
    from chronos.ops import hybrid as hops, hybrid_ref as ref

    hops.load()
    H, G, D, BS = 8, 2, 128, 16
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + window)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g).bfloat16()  # noqa: E731
    B, mb = len(lens), -(-max(lens) // BS)
    kc, vc = rnd(1 + B * mb, BS, G, D), rnd(1 + B * mb, BS, G, D)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    bt = 1 + torch.randperm(B * mb, device=DEV, generator=g).int().view(B, mb)
    qkv, sink, gate = rnd(B, (H + 2 * G) * D), torch.randn(H, device=DEV, generator=g), torch.randn(B, H, device=DEV, generator=g)
    at = (bt, i32(list(range(B + 1))), i32([n - 1 for n in lens]))
    got = hops.window_attention(qkv, kc, vc, *at, sink, gate, D ** -0.5, window, keep, H, torch.bfloat16, 1)
    want = ref.window_attention(qkv.float(), kc.float(), vc.float(), *at, sink, gate, D ** -0.5, window, keep, H, torch.float32)
    # the result's rounding to bfloat16 (2^-9 of a value at most); weights to 2^-17 of theirs
    assert float((got.float().view(B, -1) - want.view(B, -1)).norm() / want.norm()) < 2.0 ** -8
