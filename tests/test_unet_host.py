"""The U-Net kernels' host side: sizes, no kernel runs here."""
from __future__ import annotations

import pytest

from sweep_amd import _core


@pytest.mark.parametrize("H,W,cin,cout", [(48, 144, 256, 256), (24, 72, 512, 512), (384, 1152, 32, 32), (7, 5000, 40, 520),
                                          (24, 72, 2048, 2048)])
def test_wgrad_scratch_is_bounded_in_the_batch(H, W, cin, cout):
    """The weight gradient's partial tiles are at most 512 of 64 x 64 channels
    and 9 taps, however many images there are, or one for each channel tile."""
    q = _core.load().swp_nn_conv_wgrad_scratch
    tiles = -(-cin // 64) * -(-cout // 64)
    bias = 512 * cout
    for N in (1, 2, 16, 64, 1000):
        assert 9 * cin * cout + bias <= int(q(N, H, W, cin, cout, 3)) <= max(512, tiles) * 9 * 64 * 64 + bias
