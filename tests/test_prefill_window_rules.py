"""The rules that say in how many windows the w2 pass of the tile kernels cuts a reduction: what they never do (no GPU needed)."""
import pytest
import torch  # noqa: F401  (the library shares torch's HIP runtime)

from promoe_amd import _lib as L

FMTS = [L.FMT_INT4_G128, L.FMT_Q4K, L.FMT_BF16]
TOKENS = [1, 64, 65, 128, 129, 256, 257, 512, 1000, 2048, 4096]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("H", [256, 2048, 4096])
def test_shared_windows(fmt, H):
    """Pieces the entry takes, never more than the workspace is made for; a bf16 shared expert that is no longer than the routed
    experts is never cut past 64 tokens."""
    for T in TOKENS:
        for I in (128, 1408, 2816, 4096, 5632, 14336):
            for I_sh in (128, 1408, 2048, 2816, 4096, 5120, 5632, 20480):
                if fmt == L.FMT_Q4K and I_sh % 256:
                    continue
                s, most = L.lib.moe_prefill_shared_windows_beside(fmt, T, H, I, I_sh), L.lib.moe_prefill_shared_windows(fmt, T, H, I_sh)
                assert s in (1, 2, 4, 8) and s <= most, (T, I, I_sh)
                if s > 1:
                    per = I_sh // 64 // s
                    assert I_sh // 64 % s == 0 and per >= 2, (T, I, I_sh, s)
                    if fmt == L.FMT_BF16 and T > 64:
                        assert per % 2 == 0 and I_sh > I, (T, I, I_sh, s)


@pytest.mark.parametrize("fmt", FMTS)
def test_routed_windows(fmt):
    """Whole windows of at least 32 slabs, bf16 none; a launch that has a workgroup for every place of the chip (512) is cut only
    where the windows stay long."""
    for T in TOKENS:
        for E, k in ((4, 2), (8, 2), (16, 2), (32, 4), (64, 6), (128, 8)):
            for H in (256, 2048, 4096):
                for I in (128, 1408, 4096, 6144, 8192, 14336):
                    s, nk = L.lib.moe_prefill_routed_windows(fmt, T, k, E, H, I), I // 64
                    assert s in (1, 2, 4) and (s == 1 or (fmt != L.FMT_BF16 and nk % s == 0 and nk // s >= 32)), (T, E, H, I)
                    if s > 1 and nk // s < 96:
                        assert (min(T * k, E) + T * k // 128) * (H // 256) * s // 2 <= 512, (T, E, H, I, s)
