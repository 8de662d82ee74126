"""Blocks that fit the library's static array (64 MiB) on few partial sums of the down projection keep fitting: a plan that
splits the reduction further is not taken where it alone would take the block past that.  A block that is past it either way
may split further; its workspace stays small against the weights that it reads (CPU only)."""
import ctypes as C

import pytest

from on_device_sd_amd import _lib


def _workspace(T, H, I, E, K):
    s = _lib.MoeShape(T, H, E, K, I, 1, _lib.DT_BF16, 0)
    return _lib.load().odsd_moe_workspace_bytes(C.byref(s))


# (each needs 70 to 102 MB when the reduction is split as far as the equal-share kernel would)
@pytest.mark.parametrize("T,H,I,E,K", [(1000, 2048, 4096, 256, 2), (256, 2048, 8192, 256, 8), (160, 2048, 14336, 128, 8),
                                       (300, 4096, 4096, 256, 8), (300, 2048, 3584, 256, 8), (512, 4096, 5632, 128, 1),
                                       (100, 3072, 18432, 128, 8), (1500, 2048, 2304, 256, 2)])
def test_workspace_stays_within_the_static_array(T, H, I, E, K):
    assert 0 < _workspace(T, H, I, E, K) <= 64 << 20


@pytest.mark.parametrize("T,H,I,E,K", [(512, 4096, 14336, 512, 8), (768, 4096, 14336, 128, 2), (512, 4096, 5632, 512, 8)])
def test_workspace_past_the_static_array_is_small_against_the_weights(T, H, I, E, K):
    ws = _workspace(T, H, I, E, K)
    assert 64 << 20 < ws <= 0.04 * E * 1.59375 * H * I
