"""The narrowest MEX kernels, which the FP32 form takes alone (up to 3 pixels), and
the next ones, against the FP64 oracle; segment calls against per-slice calls.

Tolerance: sums of at most 49 terms, rounded 49 times to 2^-24 of the sum of their
sizes: 2.9e-6.
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [1, 3, 5, 7])
@pytest.mark.parametrize("W,H,n", [(1, 1, 1), (14, 17, 3), (481, 5, 9), (150, 31, 8)])
def test_narrow_kernels(W, H, n, kw):
    rng = np.random.default_rng(kw)
    b = rng.random((W, H, n)).astype(np.float32)
    K = (rng.random((kw, kw, 15, 15)) - 0.3).astype(np.float32)
    got = mesolf_amd.mex_lfm_convolution_vec(b, K)
    ref = O.mex_op(b.astype(np.float64), K.astype(np.float64))
    size = O.mex_op(b.astype(np.float64), np.abs(K).astype(np.float64))
    assert np.abs(got - ref).max() <= 2.9e-6 * size.max()
    K2 = np.stack([K, K[::-1]], axis=-1)
    plane, ptr = np.arange(n, dtype=np.int32) % 2, np.array([0, (n + 1) // 2, n], np.int64)
    seg = mesolf_amd.lfm_convolution_segments(b, plane, ptr, K2)
    for s in range(2):
        sum_ = np.zeros((W, H), np.float32)
        for z in range(2):
            for i in range(ptr[s], ptr[s + 1]):
                if plane[i] == z:
                    sum_ = sum_ + mesolf_amd.mex_lfm_convolution_vec(b[:, :, i:i + 1], K2[..., z])[:, :, 0]
        assert np.array_equal(seg[:, :, s], sum_)
