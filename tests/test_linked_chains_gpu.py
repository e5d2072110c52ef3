"""The chains whose neighbouring 128-row blocks are coupled through precomputed links
(lucid_link_kernel), at the block counts where the coupling can go wrong: one block (no link),
two (a link and nothing swept), three (one pair or block taken apart), four (the first full
sweep step) and more, ragged ends, both chain precisions in one call, head dims with padded
columns, fp32; and the lengths at which the forward and the backward change kernels (MHA at
head dim 64 below and from T = 2048, head dim 128 at odd multiples of 128).  Against float64
(oracle.lucid_ref.lucid_group_torch) with the bars of tests/bars.py."""
import pytest
import torch

from bars import check, check_f32
from oracle import lucid_ref as R

pytestmark = pytest.mark.gpu


def _run(B, Hq, Hkv, T, d, dtype, shared, noise=0.5):
    from lucid_amd import lucid_attention

    g = torch.Generator().manual_seed(T + d + Hq)
    q, k, v, do = (torch.randn(B, T, h, d, generator=g) for h in (Hq, Hkv, Hkv, Hq))
    if shared:  # the first kv head's keys along a direction: the exact chains
        k[:, :, 0] = (torch.randn(d, generator=g) + noise * k[:, :, 0]) / (1 + noise ** 2) ** 0.5
    q, k, v, do = (x.to(dtype).cuda() for x in (q, k, v, do))
    leaves = [x.transpose(1, 2).detach().requires_grad_() for x in (q, k, v)]
    print(f"case linked B={B} Hq={Hq} Hkv={Hkv} T={T} d={d} {dtype} shared={shared}", flush=True)
    o, vp = lucid_attention(*leaves, return_vprime=True)
    o.backward(do)
    torch.cuda.synchronize()
    G = Hq // Hkv
    chk = check_f32 if dtype == torch.float32 else check
    for b in range(B):
        for h in range(Hkv):
            hs = slice(h * G, h * G + G)
            ref = R.lucid_group_torch(leaves[0][b, hs].detach(), leaves[1][b, h].detach(), leaves[2][b, h].detach(),
                                      do[b, :, hs].transpose(0, 1))
            got = {"vp": vp[b, h], "o": o[b, :, hs].transpose(0, 1), "dq": leaves[0].grad[b, hs],
                   "dk": leaves[1].grad[b, h], "dv": leaves[2].grad[b, h]}
            for n, x in got.items():
                err, scale = (x.double() - ref[n]).abs().max().item(), ref[n].abs().max().item()
                chk(f"{n}[{b},{h}]", err, scale)
                if n == "vp" and dtype == torch.bfloat16:  # fp32 accumulation: far below the bf16 bar
                    assert err <= 4e-3 * max(1.0, scale), (n, err, scale)


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("T", [100, 128, 256, 300, 384, 512, 640, 1152])
@pytest.mark.parametrize("d", [64, 128])
def test_block_counts(T, d, shared):
    _run(1, 4, 2, T, d, torch.bfloat16, shared)


@pytest.mark.parametrize("T", [128, 256, 384, 640])
@pytest.mark.parametrize("d", [64, 68, 96, 128])
def test_block_counts_fp32(T, d):
    _run(1, 2, 2, T, d, torch.float32, False)


@pytest.mark.parametrize("B,H,T,d", [(2, 2, 1920, 64), (2, 2, 2048, 64), (1, 3, 2100, 64), (1, 2, 2176, 128),
                                     (1, 20, 2048, 64), (1, 2, 1152, 80)])
@pytest.mark.parametrize("shared", [False, True])
def test_lengths_where_the_kernels_change(B, H, T, d, shared):
    _run(B, H, H, T, d, torch.bfloat16, shared)


def test_256_column_chain():
    """The 256-column backward chain serves many long heads only."""
    _run(1, 16, 16, 32768, 64, torch.bfloat16, True)


def test_256_row_chain_at_head_dim_128():
    _run(1, 96, 96, 4352, 128, torch.bfloat16, False)
