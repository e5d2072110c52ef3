"""Launches of a forward: the coupling of the chain blocks (lucid_zx_link_kernel) takes one launch
where it need not wait for the head masses (a single 128-row block, a forced precision, fp32), two
otherwise, and short or crowded calls at head dim 128 keep the 256-row chain.  The joined launch
against float64 as in test_linked_chains_gpu."""
import ctypes

import pytest
import torch

from test_linked_chains_gpu import _run

pytestmark = pytest.mark.gpu


def _kernels(B, Hq, Hkv, T, d, dtype, precision="auto"):
    """Launch counts by kernel name of one forward."""
    from lucid_amd import _lib, lucid_attention
    from lucid_amd.lucid import precision as forced

    g = torch.Generator().manual_seed(T)
    q, k, v = (torch.randn(B, h, T, d, generator=g).to(dtype).cuda() for h in (Hq, Hkv, Hkv))
    lib = _lib.load()
    print(f"case launches B={B} Hq={Hq} Hkv={Hkv} T={T} d={d} {dtype} {precision}", flush=True)
    with forced(precision), torch.no_grad():
        lib.lucid_profile_reset()
        lib.lucid_profile_enable(1)
        try:
            lucid_attention(q, k, v)
        finally:
            lib.lucid_profile_enable(0)
        n = lib.lucid_profile_collect()
        out = {}
        for i in range(n):
            name, ms, cnt = ctypes.create_string_buffer(256), ctypes.c_double(), ctypes.c_long()
            assert lib.lucid_profile_entry(i, name, 256, ctypes.byref(ms), ctypes.byref(cnt)) == 0
            out[name.value.decode()] = cnt.value
        lib.lucid_profile_reset()
    return out


@pytest.mark.parametrize("Hq,Hkv,T,d,dtype,precision", [
    (2, 2, 128, 64, torch.bfloat16, "auto"), (4, 2, 128, 64, torch.bfloat16, "auto"),
    (4, 2, 128, 128, torch.bfloat16, "auto"), (2, 2, 512, 64, torch.bfloat16, "exact"),
    (4, 2, 384, 128, torch.bfloat16, "fast"), (2, 2, 512, 64, torch.float32, "auto"),
    (2, 2, 128, 128, torch.float32, "auto"), (2, 2, 512, 64, torch.bfloat16, "fast")])
def test_one_launch_couples_the_blocks(Hq, Hkv, T, d, dtype, precision):
    got = _kernels(1, Hq, Hkv, T, d, dtype, precision)
    assert sum(n for k, n in got.items() if "_zx_" in k or "_link_" in k) == 1, got


@pytest.mark.parametrize("B,H,T,wide", [(1, 2, 256, True), (1, 2, 512, True), (1, 2, 768, False), (1, 2, 640, False),
                                        (8, 16, 1024, True), (4, 16, 1024, False), (3, 16, 2048, False),
                                        (2, 16, 8192, True)])
def test_rows_a_block_at_head_dim_128(B, H, T, wide):
    got = _kernels(B, H, H, T, 128, torch.bfloat16)
    assert ("lucid_precond_fwd_wide_kernel" in got) == wide, got


@pytest.mark.parametrize("precision", ["exact", "fast"])
@pytest.mark.parametrize("T", [128, 256, 384, 1152])
@pytest.mark.parametrize("Hq,Hkv,d", [(2, 2, 64), (4, 2, 64), (4, 2, 128)])
def test_forced_precision(Hq, Hkv, T, d, precision):
    from lucid_amd.lucid import precision as forced

    with forced(precision):
        _run(1, Hq, Hkv, T, d, torch.bfloat16, precision == "exact")


@pytest.mark.parametrize("shared", [False, True])
def test_one_block_of_many_heads(shared):
    """Each workgroup decides by its own head's mass (one launch, exact heads among the others)."""
    _run(2, 20, 20, 128, 64, torch.bfloat16, shared)
    _run(2, 20, 10, 100, 64, torch.bfloat16, shared)


@pytest.mark.parametrize("T", [256, 512])
@pytest.mark.parametrize("d", [64, 128])
def test_crowded_short_calls(d, T):
    """Many short heads: the 256-row and the 256-column chains, from one block of each on."""
    _run(5, 17, 17, T, d, torch.bfloat16, True)
