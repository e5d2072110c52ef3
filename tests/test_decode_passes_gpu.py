"""Decoding calls of several tokens at the counts where the passes change: one 32-column score
tile, two of them (groups of 4 and 8), the last pass shorter than the others, and the fewest and
most cached rows of a split (one row, a tile's remainder, many splits merged four at a time).
Against the definition in float64, with the bars of tests/bars.py."""
import pytest
import torch

from bars import check

pytestmark = pytest.mark.gpu


def _reference(q, k, v, kc, vc, eps=1e-5):
    q, k, v, kc, vc = (x.double() for x in (q, k, v, kc, vc))
    B, Hq, L, d = q.shape
    Hkv, n, s = k.shape[1], kc.shape[2], d ** -0.5
    keys = torch.cat([kc, k], 2)
    kh = keys * torch.rsqrt(keys.pow(2).mean(-1, keepdim=True) + eps)
    vps = torch.cat([vc, torch.zeros_like(v)], 2)
    o = torch.empty(B, L, Hq, d, dtype=torch.float64, device=q.device)
    for t in range(L):
        m = n + t
        p = torch.exp(s * (kh[:, :, m:m + 1] * kh[:, :, :m + 1]).sum(-1) - 1 / s)
        vps[:, :, m] = (v[:, :, t] - (p[..., :m, None] * vps[:, :, :m]).sum(2)) / p[..., m:]
        sc = s * (q[:, :, t].reshape(B, Hkv, -1, 1, d) * keys[:, :, None, :m + 1]).sum(-1)
        o[:, t] = (torch.softmax(sc, -1)[..., None] * vps[:, :, None, :m + 1]).sum(3).reshape(B, Hq, d)
    return o, vps[:, :, n:]


@pytest.mark.parametrize("d", [64, 68, 128])
@pytest.mark.parametrize("G,L", [(1, 1), (1, 17), (2, 11), (3, 9), (4, 1), (4, 6), (4, 7), (4, 12), (4, 13), (4, 25),
                                 (8, 1), (8, 3), (8, 4), (8, 7), (8, 8), (8, 15)])
@pytest.mark.parametrize("n", [1, 70, 2300])
def test_passes(G, L, d, n):
    from lucid_amd.lucid import lucid_decode

    B, Hkv = 2, 2
    g = torch.Generator(device="cuda").manual_seed(G * L + d + n)
    dp = 64 if d <= 64 else 128
    kc, vc = (torch.zeros(B, Hkv, n + L + 3, dp, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    for c in (kc, vc):
        c[:, :, :n, :d] = torch.randn(B, Hkv, n, d, generator=g, device="cuda")
    q, k, v = (torch.randn(B, L, h, d, generator=g, device="cuda").to(torch.bfloat16).transpose(1, 2)
               for h in (G * Hkv, Hkv, Hkv))
    ro, rv = _reference(q, k, v, kc[:, :, :n, :d], vc[:, :, :n, :d])
    print(f"case decode G={G} L={L} d={d} n={n}", flush=True)
    o, vp = lucid_decode(q, k, v, kc, vc, n)
    torch.cuda.synchronize()
    check("o", (o.double() - ro).abs().max().item(), ro.abs().max().item())
    check("vp", (vp.double() - rv).abs().max().item(), rv.abs().max().item())
    assert torch.equal(kc[:, :, n:n + L, :d], k) and torch.equal(vc[:, :, n:n + L, :d], vp.to(torch.bfloat16))
    assert not kc[:, :, n + L:].any() and not vc[:, :, n + L:].any()
