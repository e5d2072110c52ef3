"""Workspace sizes: those of the padded head dim, never smaller for a longer sequence or a larger
batch (a buffer sized once for the largest call serves the others), and large enough for the
shares of a split dK/dV' sweep.  The queries are host functions; nothing is launched."""
import pytest

ATTN = ("lucid_fwd", "lucid_bwd", "lucid_fwd_f32", "lucid_bwd_f32", "lucid_attn_vp_fwd", "lucid_attn_vp_fwd_f32",
        "lucid_attn_vp_bwd", "lucid_attn_vp_bwd_f32")
HEADS = [(16, 16), (8, 8), (32, 8), (32, 4), (12, 4), (4, 1), (32, 1)]


def _size(name):
    from lucid_amd import _lib

    return getattr(_lib.load(), f"{name}_workspace_bytes")


@pytest.mark.parametrize("B,Hq,Hkv,T,D", [(0, 1, 1, 128, 64), (1, 1, 1, 0, 64), (1, 1, 1, 64, 128), (1, 0, 0, 128, 64)])
def test_zero_sizes(B, Hq, Hkv, T, D):
    """Queries return for any sizes, zero included: at most the smallest launchable size's bytes."""
    for name in ATTN:
        assert _size(name)(B, Hq, Hkv, T, D) <= _size(name)(max(B, 1), max(Hq, 1), max(Hkv, 1), 128, D), name
    assert _size("lucid_precond_bwd")(B, Hkv, T, D) <= _size("lucid_precond_bwd")(max(B, 1), max(Hkv, 1), 128, D)


@pytest.mark.parametrize("name", ATTN)
@pytest.mark.parametrize("Hq,Hkv", HEADS)
def test_sizes_are_those_of_the_padded_head_dim(name, Hq, Hkv):
    size = _size(name)
    for T in (128, 256, 896, 1024, 2048, 4096, 8064, 8192, 16256, 32768):
        for B in (1, 2, 8):
            for dims in ((1, 32, 63, 64), (65, 68, 80, 96, 97, 100, 128)):
                got = {size(B, Hq, Hkv, T, d) for d in dims}
                assert len(got) == 1, (T, B, dims, got)


@pytest.mark.parametrize("name", ATTN)
@pytest.mark.parametrize("Hq,Hkv", HEADS)
def test_sizes_never_fall(name, Hq, Hkv):
    size = _size(name)
    for D in (64, 96, 128):
        for B in (1, 2, 3, 4, 8):
            over_t = [size(B, Hq, Hkv, T, D) for T in range(128, 32768 + 1, 128)]
            assert all(a <= b for a, b in zip(over_t, over_t[1:])), (D, B)
        for T in (128, 1024, 4096, 8192, 16000, 32768):
            over_b = [size(B, Hq, Hkv, T, D) for B in range(1, 33)]
            assert all(a <= b for a, b in zip(over_b, over_b[1:])), (D, T)


def _shares(B, Hq, Hkv, T, D, f32):
    """Shares of a column block in the dK/dV' sweep: two workgroups per slot, at least eight
    64-row steps in the longest share, at most eight shares (dkdv_splits in lucid_capi.hip)."""
    wide = not f32 and D > 64 and T >= (1024 if D <= 96 else 8192)
    jobs = B * Hkv * (-(-T // 256) if wide else T // 128)
    slots = 512 if D <= 64 and not f32 else 256
    return max(1, min(8, -(-2 * slots // jobs), Hq // Hkv * (T // 64) // 8))


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("Hq,Hkv", HEADS)
def test_the_partial_sums_fit(Hq, Hkv, f32):
    """The attention seam's scratch holds dV', delta, its seeds, dK, (fp32: the pair of dO) and
    the counters beside the partial sums, nothing else."""
    size = _size("lucid_attn_vp_bwd" + ("_f32" if f32 else ""))
    split = 0
    for B in (1, 2, 4, 8):
        for T in (*range(128, 4096, 128), 4096, 8064, 8192, 16000, 16256, 16384, 32640, 32768):
            for D in (64, 68, 96, 128):
                dp = 64 if D <= 64 else 128
                rows, qrows, n = B * Hkv * T, B * Hq * T, _shares(B, Hq, Hkv, T, D, f32)
                base = 8 * rows * dp + qrows * (36 + (4 * dp if f32 else 0))
                assert size(B, Hq, Hkv, T, D) >= base + (n - 1) * 8 * rows * dp, (B, T, D, n)
                split += n > 1
    assert split > 20
