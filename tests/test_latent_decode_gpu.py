"""Latent attention of decode rows at the edges of its key tiles, its rounds of tiles on the way and of looked-up rows, against
float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,DK,rank", [(16, 576, 512), (32, 576, 512), (17, 536, 496), (7, 320, 256), (32, 328, 288), (20, 304, 256)])
@pytest.mark.parametrize("B,two_term,window,sink", [(9, False, 0, False), (9, True, 0, True), (40, False, 90, False),
                                                    (260, False, 0, True)])
def test_latent_decode_tiles(H, DK, rank, B, two_term, window, sink):
    """260 sequences are served without a split of the keys: the one of 2600 keys walks 82 tiles and looks rows up three times.  Bound, per
    element and with the weights w: the softmax weights are rounded once (bfloat16 has 8 significant bits: half a unit in the last place is at
    most 2^-8 of a value, in two terms 2^-16), the output once (2^-8 |o|); a score is off by at most
    DK 2^-24 of the sum of its products' sizes, which moves a weight by twice that."""
    from chronos.ops import hybrid as hops

    g = torch.Generator().manual_seed(H + DK + B)
    BS = 16
    edges = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 192, 193]
    lens = [2600] + [edges[(b * 7 + H) % len(edges)] for b in range(B - 1)]
    pages = [(n + BS - 1) // BS for n in lens]
    perm = (torch.randperm(sum(pages), generator=g) + 1).int()
    bt = torch.zeros(B, max(pages) + 2, dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        bt[b, :n] = perm[at:at + n]
        at += n
    cache = torch.randn(sum(pages) + 1, BS, DK, generator=g).bfloat16()
    qa = torch.randn(B, H, DK, generator=g).bfloat16()
    sk = torch.randn(H, generator=g) if sink else None
    scale = DK ** -0.5
    q_start = torch.arange(B + 1, dtype=torch.int32)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32)
    d = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    out = hops.latent_attention(d(qa), d(cache), d(bt), d(q_start), d(pos), None, scale, rank, torch.bfloat16, 1, window, two_term, d(sk))
    qa, cache, out = qa.to(DEV).double(), cache.to(DEV), out.double()
    for b, n in enumerate(lens):
        keys = cache[bt[b, :pages[b]].long().to(DEV)].flatten(0, 1)[:n].double()
        lo = max(0, n - window) if window else 0
        keys = keys[lo:]
        s = qa[b] @ keys.T * scale                                            # [H, n]
        ds = (DK * 2.0 ** -24 * (qa[b].abs() @ keys.abs().T) * scale).amax(-1, keepdim=True)
        m = s.amax(-1, keepdim=True)
        if sink:
            m = torch.maximum(m, sk.to(DEV).double()[:, None])
        e = (s - m).exp()
        den = e.sum(-1, keepdim=True) + ((sk.to(DEV).double()[:, None] - m).exp() if sink else 0)
        w = e / den
        want, size = w @ keys[:, :rank], w @ keys[:, :rank].abs()
        bound = (2.0 ** (-16 if two_term else -8) + 2 * ds + 2.0 ** -18) * size + 2.0 ** -8 * want.abs() + 1e-30
        bad = ((out[b] - want).abs() > bound).nonzero()
        assert bad.numel() == 0, (b, n, bad[:4].tolist())
