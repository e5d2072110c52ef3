"""Workspace queries return for any sizes, zero included (they take none of the launches' checks)."""
import pytest


@pytest.mark.parametrize("B,Hq,Hkv,T,D", [(0, 1, 1, 128, 64), (1, 1, 1, 0, 64), (1, 1, 1, 64, 128), (1, 0, 0, 128, 64)])
def test_zero_sizes(B, Hq, Hkv, T, D):
    from lucid_amd import _lib

    lib = _lib.load()
    for name in ("lucid_fwd", "lucid_bwd", "lucid_fwd_f32", "lucid_bwd_f32", "lucid_attn_vp_bwd", "lucid_attn_vp_bwd_f32"):
        assert getattr(lib, f"{name}_workspace_bytes")(B, Hq, Hkv, T, D) >= 0
    assert lib.lucid_precond_bwd_workspace_bytes(B, Hkv, T, D) >= 0
