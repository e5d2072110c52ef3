"""lucid_pad_rows (the zero-padding of a call's operands) against torch.nn.functional.pad, bit for
bit: rows that start at any element alignment, columns that end inside a 16-byte chunk, one to
three tensors of different head counts, views and expanded tensors, and no padding at all."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,tp", [(1, 128), (127, 128), (128, 128), (5, 5)])
@pytest.mark.parametrize("d,dp", [(1, 64), (63, 64), (64, 64), (66, 128), (68, 128), (127, 128)])
def test_matches_torch_pad(T, tp, d, dp, dtype):
    from lucid_amd.lucid import _pad_rows

    B = 2
    g = torch.Generator(device="cuda").manual_seed(T * d)
    qkv = torch.randn(B, T, 3, 3 * d + 1, generator=g, device="cuda").to(dtype)  # odd row offsets
    ts = [qkv[..., i * d:i * d + d].transpose(1, 2)[:, :h] for i, h in enumerate((3, 1, 2))]
    for n in (1, 2, 3):
        for x, y in zip(ts[:n], _pad_rows(ts[:n], tp, dp)):
            assert y.is_contiguous() and torch.equal(y, F.pad(x, (0, dp - d, 0, tp - T)))
    e = torch.randn(1, 1, 1, d, device="cuda").to(dtype).expand(B, 2, T, d)
    assert torch.equal(_pad_rows((e,), tp, dp)[0], F.pad(e, (0, dp - d, 0, tp - T)))
    w = torch.randn(B, 2, d, T, device="cuda").to(dtype).transpose(2, 3)  # no unit stride
    assert torch.equal(_pad_rows((w,), tp, dp)[0], F.pad(w, (0, dp - d, 0, tp - T)))


@pytest.mark.parametrize("T,d,dtype", [(100, 64, torch.bfloat16), (128, 40, torch.bfloat16), (130, 68, torch.float32)])
def test_gradients_of_a_padded_call_reach_strided_leaves(T, d, dtype):
    """The padding is inside the autograd step: O, V' and the gradients have the caller's shapes."""
    from lucid_amd import lucid_attention

    x = torch.randn(1, T, 4, d, device="cuda").to(dtype).requires_grad_()
    k = torch.randn(1, T, 2, d, device="cuda").to(dtype).requires_grad_()
    v = torch.randn(1, T, 2, d, device="cuda").to(dtype).requires_grad_()
    o, vp = lucid_attention(x.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), return_vprime=True)
    assert o.shape == (1, T, 4, d) and vp.shape == (1, 2, T, d)
    o.sum().backward()  # an expanded gradient
    for leaf in (x, k, v):
        assert leaf.grad.shape == leaf.shape and torch.isfinite(leaf.grad).all()
    g0 = [t.grad.clone() for t in (x, k, v)]
    x.grad = k.grad = v.grad = None
    pad = (0, 0, 0, 128 - T % 128 if T % 128 else 0)  # the same call on keys padded by hand
    o2 = lucid_attention(*(F.pad(t.transpose(1, 2), pad) for t in (x, k, v)))
    o2[:, :T].sum().backward()
    assert torch.equal(o2[:, :T], o)
    for a, b in zip(g0, (x, k, v)):
        assert torch.equal(a, b.grad)
