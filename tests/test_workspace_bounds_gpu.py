"""The backward stays inside workspaces sized the ways the C header allows: by the padded head dim
for a smaller one, and by the longest sequence or the largest batch for the others.  The workspace
lies in a larger allocation whose remainder must keep its pattern, and the gradients are those of
a workspace of the call's own size."""
import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 96 << 20


# (B, Hq, Hkv, T, d) of the call, of the sizes the workspace is made for; the shares of the dK/dV'
# sweep differ between the two
@pytest.mark.parametrize("call,sized", [
    ((1, 32, 8, 4096, 96), (1, 32, 8, 4096, 128)),
    ((1, 32, 4, 2048, 68), (1, 32, 4, 2048, 128)),
    ((1, 16, 16, 8064, 64), (1, 16, 16, 8192, 64)),
    ((1, 32, 8, 8064, 128), (1, 32, 8, 8192, 128)),
    ((1, 32, 4, 2048, 64), (8, 32, 4, 2048, 64)),
    ((1, 4, 1, 128, 64), (1, 4, 1, 4096, 64)),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_in_a_workspace_of_other_sizes(call, sized, dtype):
    from lucid_amd import _lib
    from lucid_amd import lucid as L

    lib = _lib.load()
    B, Hq, Hkv, T, d = call
    f32 = dtype == torch.float32
    print(f"case workspace bounds call={call} sized={sized} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + d)
    dp = 64 if d <= 64 else 128
    q, k, v, do = (torch.zeros(B, h, T, dp, dtype=dtype, device="cuda") for h in (Hq, Hkv, Hkv, Hq))
    for x in (q, k, v, do):
        x[..., :d] = torch.randn(*x.shape[:3], d, generator=g, device="cuda").to(dtype)
    dot = do.transpose(1, 2)
    scale, eps = d ** -0.5, 1e-5
    if f32:
        o, _, lse, ws = L._fwd_f32(q, k, v, scale, eps, d)
        ref = L._bwd_f32(dot, Hkv, o, lse, ws, scale, d)
    else:
        o, _, lse, ws = L._fwd(q, k, v, scale, eps, d)
        ref = L._bwd(dot, q, k, o, lse, ws, scale, eps, d)
    n = (lib.lucid_bwd_f32_workspace_bytes if f32 else lib.lucid_bwd_workspace_bytes)(*sized)
    buf = torch.full((n + GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
    got = [torch.empty_like(x) for x in (q, k, v)]
    p, s = _lib.ptr, lambda t: _lib.strides3(t, (0, 1, 2))
    head = (p(dot), _lib.strides3(dot, (0, 2, 1)))
    tail = (p(o), _lib.strides3(o, (0, 2, 1)), p(lse), p(ws), *(a for t in got for a in (p(t), s(t))), p(buf), *call, scale)
    st = _lib.stream_handle(q.device)
    if f32:
        rc = lib.lucid_attn_bwd_f32(*head, *tail, st)
    else:
        rc = lib.lucid_attn_bwd(*head, p(q), s(q), p(k), s(k), *tail, eps, st)
    _lib.check(lib, rc, "backward")
    torch.cuda.synchronize()
    assert bool((buf[n:] == 0xA5).all()), "written past the workspace"
    for a, b in zip(got, ref):
        assert torch.equal(a, b.reshape(a.shape))
