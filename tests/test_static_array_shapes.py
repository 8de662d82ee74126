"""Blocks that fit the library's static array (64 MiB) on few partial sums of the down projection keep fitting: a plan that
splits the reduction further is not taken where it alone would take the block past that (CPU only)."""
import ctypes as C

import pytest

from on_device_sd_amd import _lib


@pytest.mark.parametrize("T,H,I,E,K", [(1000, 2048, 4096, 256, 2), (256, 2048, 8192, 256, 8), (160, 2048, 14336, 128, 8),
                                       (300, 4096, 4096, 256, 8), (600, 4096, 8192, 128, 2), (48, 4096, 14336, 8, 2)])
def test_workspace_stays_within_the_static_array(T, H, I, E, K):
    s = _lib.MoeShape(T, H, E, K, I, 1, _lib.DT_BF16, 0)
    assert 0 < _lib.load().odsd_moe_workspace_bytes(C.byref(s)) <= 64 << 20
