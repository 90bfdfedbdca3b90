"""The BF16 split form of the MEX operator (mex_split.hip) at its edges.

Tolerance against the FP64 oracle: a product leaves out three partial products
of at most 2^-24 of it each, and a sum of m terms is rounded 6 m / 32 times to
2^-24 of the partial sum.  With kernels up to 61 wide (m = 61 * 80) those are
about 920 roundings of random sign, sqrt(920) * 2^-24 = 1.8e-6 relative at
most; 2e-6 is asked for.
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


def _inputs(W, H, n, kw, seed=3):
    rng = np.random.default_rng(seed)
    b = (rng.random((W, H, n)) * (rng.random((W, H, n)) < 0.3)).astype(np.float32)
    K = (rng.random((kw, kw, 15, 15)) - 0.2).astype(np.float32)
    return b, K


# widths around whole lenslets; image counts that end M blocks early, exactly and
# late; kernels of one lenslet pair, odd and even pair counts, wider than the bitmap
@pytest.mark.parametrize("W,H,n,kw", [
    (1, 1, 1, 1), (14, 3, 2, 3), (15, 16, 1, 15), (16, 15, 3, 17), (31, 29, 7, 29), (45, 17, 16, 31),
    (46, 5, 40, 33), (90, 7, 86, 43), (47, 61, 2, 61), (20, 9, 3, 59), (225, 6, 35, 13), (61, 4, 130, 9),
])
def test_split_form_against_the_oracle(W, H, n, kw):
    b, K = _inputs(W, H, n, kw)
    got = mesolf_amd.mex_lfm_convolution_vec(b, K)
    ref = O.mex_op(b.astype(np.float64), K.astype(np.float64))
    # cancelling taps: compared with the sum of the terms' sizes
    size = O.mex_op(np.abs(b).astype(np.float64), np.abs(K).astype(np.float64))
    assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(size), rel_l2(got, ref)


def test_split_form_scales_exactly():
    """Powers of two change no significand, so the result scales bit for bit."""
    b, K = _inputs(47, 33, 3, 31)
    one = mesolf_amd.mex_lfm_convolution_vec(b, K)
    for e in (-60, 80):
        assert np.array_equal(mesolf_amd.mex_lfm_convolution_vec(np.ldexp(b, e).astype(np.float32), K),
                              np.ldexp(one, e).astype(np.float32)), e


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.finfo(np.float32).max])
@pytest.mark.parametrize("where", ["bitmap", "kernel"])
def test_values_that_bf16_cannot_hold(value, where):
    """A non-finite (or BF16-overflowing) value reaches only what the FP32 form
    lets it reach: outputs whose padded window misses it stay as they are, an
    infinity stays one, and the next call is unaffected."""
    W, H, n, kw = 150, 60, 3, 31
    b, K = _inputs(W, H, n, kw)
    K = np.abs(K) + np.float32(0.01)
    b[70, 30, 1] = 1.0
    clean = mesolf_amd.mex_lfm_convolution_vec(b, K)
    b2, K2 = b.copy(), K.copy()
    if where == "bitmap":
        b2[70, 30, 1] = value
        hit = np.zeros((W, H, n), bool)
        hit[70 - 15 - 14:70 + 15 + 15, 15:46, 1] = True  # taps t = kx + phase of whole lenslets
        sure = (70, 30, 1)
    else:
        K2[15, 15, 70 % 15, 0] = value  # tap of phase (10, 0), at the output's own pixel
        hit = np.zeros((W, H, n), bool)
        hit[:, 0::15, :] = True
        sure = (70, 30, 1)
    got = mesolf_amd.mex_lfm_convolution_vec(b2, K2)
    size = O.mex_op(b.astype(np.float64), K.astype(np.float64))
    assert np.abs(got - clean)[~hit].max() <= 1e-5 * size.max()
    if np.isnan(value):
        assert np.isnan(got[sure])
    elif np.isinf(value):
        assert got[sure] == value
    else:
        assert got[sure] > 1e36
    assert np.array_equal(mesolf_amd.mex_lfm_convolution_vec(b, K), clean)
