"""The fp32 solve in place: V' written over V (one contiguous buffer passed as both), as the
reference's solver does (modeling_lucid.py:296-299), gives the bytes of the solve into another
buffer.  Through the C entry points; the Python layer never passes one buffer as both."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [128, 256, 384, 512, 640, 1152])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("entry", ["tril_solve", "get_v_prime", "attn_fwd"])
def test_v_prime_over_v(entry, T, D):
    from lucid_amd import _lib

    lib = _lib.load()
    print(f"case in place {entry} T={T} D={D}", flush=True)
    B, Hq, Hkv = 2, 4, 2
    g = torch.Generator(device="cuda").manual_seed(T + D)
    q, k, v = (torch.randn(B, h, T, D, generator=g, device="cuda") for h in (Hq, Hkv, Hkv))
    if entry == "tril_solve":
        k = k * torch.rsqrt(k.pow(2).mean(-1, keepdim=True) + 1e-5)
    scale, eps, p = D ** -0.5, 1e-5, _lib.ptr
    st = _lib.stream_handle(k.device)
    size = lib.lucid_fwd_f32_workspace_bytes if entry == "attn_fwd" else lib.lucid_v_prime_f32_workspace_bytes
    ws = torch.empty(size(B, *((Hq, Hkv) if entry == "attn_fwd" else (Hkv,)), T, D), dtype=torch.uint8, device="cuda")

    def solve(v, vp):
        s = [_lib.strides3(t, (0, 1, 2)) for t in (q, k, v)]
        if entry == "tril_solve":
            rc = lib.lucid_tril_solve_f32(p(k), s[1], p(v), s[2], p(vp), p(ws), B, Hkv, T, D, scale, st)
        elif entry == "get_v_prime":
            rc = lib.lucid_get_v_prime_f32(p(k), s[1], p(v), s[2], p(vp), p(ws), B, Hkv, T, D, scale, eps, st)
        else:
            o = torch.empty(B, T, Hq, D, device="cuda")
            lse = torch.empty(B, Hq, T, device="cuda")
            rc = lib.lucid_attn_fwd_f32(p(q), s[0], p(k), s[1], p(v), s[2], p(o), _lib.strides3(o, (0, 2, 1)), p(vp),
                                        p(lse), p(ws), B, Hq, Hkv, T, D, scale, eps, st)
        _lib.check(lib, rc, entry)
        torch.cuda.synchronize()
        return vp

    want = solve(v, torch.empty_like(v))
    x = v.clone()
    assert torch.equal(solve(x, x), want)
