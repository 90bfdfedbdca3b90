"""The rectification kernel at the edges of its tiles (4 columns and 256 rows per
workgroup, 16 frames at a time) against scipy's interpolation: FP64 on both
sides and one rounding to single, within 2e-7 of the largest value."""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O

pytestmark = pytest.mark.gpu


# images of two rows, output columns 0 .. 3 past a multiple of 4, frames 1, 16, 17 and 33
@pytest.mark.parametrize("H,W,n,xc,yc,dx", [(2, 2, 33, 1.2, 0.7, 1.0), (2, 3, 16, 1.2, 0.7, 1.5),
                                             (300, 64, 17, 31.7, 150.2, 30.0), (530, 60, 2, 30.0, 261.3, 15.3),
                                             (37, 34, 1, 17.5, 12.0, 5.1)])
def test_rectify_tiles(H, W, n, xc, yc, dx):
    rng = np.random.default_rng(H + n)
    frames = (rng.random((H, W, n)) * 1000).astype(np.float32)
    got = mesolf_amd.img_rectify_mod(frames, xc, yc, 15, dx)
    want = O.rectify(frames.astype(np.float64), xc, yc, 15, dx)
    assert got.shape == want.shape
    assert np.max(np.abs(got - want)) <= 2e-7 * np.max(np.abs(want))
