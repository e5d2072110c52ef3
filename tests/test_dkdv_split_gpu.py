"""The split dK/dV' column sweep (few column blocks: each block's query steps are cut into
shares whose partial sums are added afterwards) and the exact chains' 32-row-wave kernels, at
the sizes where the cut can go wrong: a share that starts inside a query head, shares of
unequal length, the causal diagonal in the first share only, one head with no group, and the
smallest T that is split.  Against float64 (oracle.lucid_ref.lucid_group_torch), with the bars of
tests/bars.py (bf16 2e-2, fp32 1e-4 of the largest reference value)."""
import pytest
import torch

from bars import check, check_f32
from oracle import lucid_ref as R

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, T, d
    (1, 1, 1, 1024, 64),    # no group: the shares cut one head's query tiles (two shares)
    (1, 5, 1, 384, 64),     # three shares of a group of five: cuts inside query heads
    (1, 8, 2, 896, 64),
    (2, 7, 1, 640, 128),
    (1, 6, 2, 512, 80),     # zero-padded rows
    (1, 3, 1, 300, 64),     # ragged T
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("B,Hq,Hkv,T,d", CASES)
def test_split_column_sweep(B, Hq, Hkv, T, d, dtype):
    from lucid_amd import lucid_attention

    g = torch.Generator().manual_seed(T + d + Hq)
    q, k, v, do = (torch.randn(B, T, h, d, generator=g).to(dtype).cuda() for h in (Hq, Hkv, Hkv, Hq))
    # the last kv head's keys share a direction: that head runs the exact kernels (bf16)
    k[:, :, -1] = (0.3 * k[:, :, -1].float() + torch.randn(d, generator=g).cuda()).to(dtype)
    leaves = [x.transpose(1, 2).detach().requires_grad_() for x in (q, k, v)]
    print(f"case split B={B} Hq={Hq} Hkv={Hkv} T={T} d={d} {dtype}", flush=True)
    o = lucid_attention(*leaves)
    o.backward(do)
    torch.cuda.synchronize()
    G = Hq // Hkv
    chk = check_f32 if dtype == torch.float32 else check
    for b in range(B):
        for h in range(Hkv):
            hs = slice(h * G, h * G + G)
            ref = R.lucid_group_torch(leaves[0][b, hs].detach(), leaves[1][b, h].detach(), leaves[2][b, h].detach(),
                                      do[b, :, hs].transpose(0, 1))
            got = {"o": o[b, :, hs].transpose(0, 1), "dq": leaves[0].grad[b, hs], "dk": leaves[1].grad[b, h],
                   "dv": leaves[2].grad[b, h]}
            for n, x in got.items():
                chk(f"{n}[{b},{h}]", (x.double() - ref[n]).abs().max().item(), ref[n].abs().max().item())


@pytest.mark.parametrize("vp_dtype", [torch.bfloat16, torch.float32])
def test_split_column_sweep_of_the_attention_seam(vp_dtype):
    """eager_lucid_attention_forward's backward takes the same split (its scratch layout differs)."""
    from lucid_amd.lucid import eager_lucid_attention_forward

    g = torch.Generator().manual_seed(3)
    B, Hq, Hkv, T, d = 1, 4, 1, 700, 64
    q, k = (torch.randn(B, h, T, d, generator=g).to(torch.bfloat16).cuda().requires_grad_() for h in (Hq, Hkv))
    vp = torch.randn(B, Hkv, T, d, generator=g).to(vp_dtype).cuda().requires_grad_()
    do = torch.randn(B, T, Hq, d, generator=g).to(torch.bfloat16).cuda()
    o, _ = eager_lucid_attention_forward(q, k, vp)
    o.backward(do)
    qr, kr, vr = (x.detach().double().requires_grad_() for x in (q, k, vp.to(torch.bfloat16)))
    s = (d ** -0.5 * (qr @ kr.transpose(-1, -2))).masked_fill(
        ~torch.ones(T, T, dtype=torch.bool, device="cuda").tril(), float("-inf"))
    (torch.softmax(s, -1) @ vr).transpose(1, 2).backward(do.double())
    for n, x, r in (("dq", q, qr), ("dk", k, kr), ("dvp", vp, vr)):
        check(n, (x.grad.double() - r.grad).abs().max().item(), r.grad.abs().max().item())


@pytest.mark.parametrize("B,Hq,Hkv,T,d", [(1, 4, 2, 1152, 96), (1, 3, 1, 1024, 80), (2, 2, 2, 1408, 68),
                                          (1, 2, 1, 8320, 128), (1, 1, 1, 8192, 100)])
def test_256_key_column_blocks(B, Hq, Hkv, T, d):
    """Head dims above 64 at the lengths of the eight-wave sweep, with and without half a block at
    the end (T an odd multiple of 128)."""
    test_split_column_sweep(B, Hq, Hkv, T, d, torch.bfloat16)
