"""fp32 operands whose rows are read without padding (head dims that are multiples of 4): the same
bits as the padded route, which misaligned copies of the operands still take, with NaN in the
columns just behind every row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _views(x):
    """x inside a wider NaN-filled buffer (rows read whole), and as a 4-byte-aligned copy (padded)."""
    wide = torch.full((*x.shape[:3], x.shape[3] + 4), float("nan"), device="cuda")
    wide[..., :x.shape[3]] = x
    flat = torch.empty(x.numel() + 1, device="cuda")[1:].view(x.shape)
    return wide[..., :x.shape[3]], flat.copy_(x)


@pytest.mark.parametrize("d", [4, 36, 60, 68, 96, 124])
@pytest.mark.parametrize("B,Hq,Hkv,T", [(1, 2, 1, 128), (2, 2, 2, 384)])
def test_whole_rows_match_padded_rows(B, Hq, Hkv, T, d):
    from lucid_amd import lucid_attention
    from lucid_amd.lucid import _whole_rows

    g = torch.Generator().manual_seed(T + d)
    q, k, v, do = (_views(torch.randn(*s, generator=g).cuda())
                   for s in ((B, Hq, T, d), (B, Hkv, T, d), (B, Hkv, T, d), (B, T, Hq, d)))
    print(f"case whole rows B={B} Hq={Hq} Hkv={Hkv} T={T} d={d}", flush=True)
    res = []
    for i, whole in enumerate((True, False)):
        assert all(_whole_rows(x[i]) == whole for x in (q, k, v, do))
        leaves = [x[i].detach().requires_grad_() for x in (q, k, v)]
        o, vp = lucid_attention(*leaves, return_vprime=True)
        o.backward(do[i])
        res.append((o, vp, *(x.grad for x in leaves)))
    torch.cuda.synchronize()
    for n, a, b in zip(("o", "vp", "dq", "dk", "dv"), *res):
        assert torch.isfinite(a).all() and torch.equal(a, b), n
