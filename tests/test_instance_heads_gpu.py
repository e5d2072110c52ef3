"""Heads of both chain precisions in one call, in the orders and numbers at which the dense
numbering of an instance's heads (InstanceHeads) can go wrong: none of a kind, one at either end,
every second one, and more heads than one 64-lane ballot holds.  Against float64
(oracle.lucid_ref.lucid_group_torch) with the bars of tests/bars.py."""
import pytest
import torch

from bars import check
from oracle import lucid_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hkv,G,T,d", [(1, 3, 2, 384, 64), (2, 33, 1, 256, 64), (1, 131, 1, 128, 64),
                                         (1, 5, 2, 256, 128), (2, 2, 1, 2304, 64)])
@pytest.mark.parametrize("pattern", ["every second", "first", "last", "all"])
def test_mixed_heads(B, Hkv, G, T, d, pattern):
    from lucid_amd import lucid_attention

    BH = B * Hkv
    exact = {"every second": range(1, BH, 2), "first": [0], "last": [BH - 1], "all": range(BH)}[pattern]
    g = torch.Generator().manual_seed(BH + T + d)
    q, k, v, do = (torch.randn(B, T, h, d, generator=g) for h in (Hkv * G, Hkv, Hkv, Hkv * G))
    for i in exact:  # keys along a direction: the exact chains
        b, h = divmod(i, Hkv)
        k[b, :, h] = (torch.randn(d, generator=g) + 0.5 * k[b, :, h]) / 1.25 ** 0.5
    q, k, v, do = (x.to(torch.bfloat16).cuda() for x in (q, k, v, do))
    leaves = [x.transpose(1, 2).detach().requires_grad_() for x in (q, k, v)]
    print(f"case instance heads BH={BH} G={G} T={T} d={d} exact={pattern}", flush=True)
    o, vp = lucid_attention(*leaves, return_vprime=True)
    o.backward(do)
    torch.cuda.synchronize()
    for b in range(B):
        for h in range(Hkv):
            hs = slice(h * G, h * G + G)
            ref = R.lucid_group_torch(leaves[0][b, hs].detach(), leaves[1][b, h].detach(), leaves[2][b, h].detach(),
                                      do[b, :, hs].transpose(0, 1))
            got = {"vp": vp[b, h], "o": o[b, :, hs].transpose(0, 1), "dq": leaves[0].grad[b, hs],
                   "dk": leaves[1].grad[b, h], "dv": leaves[2].grad[b, h]}
            for n, x in got.items():
                check(f"{n}[{b},{h}]", (x.double() - ref[n]).abs().max().item(), ref[n].abs().max().item())
