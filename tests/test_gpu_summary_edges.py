"""The summary image at the frame counts where its passes change: tiles of 64 pixels
in 16 or 40 registers (256 | 257) and of 32 (548 | 549) in the rounds, of 32 and 16 in the
last pass (459 | 460), no tiles from 837 on, and none for few frames of a large image
(below npix / 20000 - 2).

Tolerances: backgrounds are FP64 sums of at most 3e6 terms in another order, 1e-9
of the result; the detrended movie is rounded to FP32 (2^-24) before a smoothing, a
third power and a standard deviation that loses at most two decimal digits here: 1e-5.
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

EDGES = [(9, 13, 256), (9, 13, 257), (11, 7, 459), (11, 7, 460), (5, 13, 548), (5, 13, 549), (7, 5, 836), (7, 5, 837),
         (300, 300, 2), (300, 300, 3), (500, 480, 9), (500, 480, 10)]


def _movie(npix, T):
    rng = np.random.default_rng(T)
    base = 200 + 50 * rng.random((npix, 1))
    return np.asfortranarray(rng.poisson(base * (1 + 0.3 * np.sin(np.arange(T) / 7.0))).astype(np.float32))


@pytest.mark.parametrize("h,w,T", EDGES)
def test_pixelwise(h, w, T):
    m = _movie(h * w, T)
    w1, w2 = max(1, min(100, T // 2)), max(1, min(20, T // 4))
    img, bs, bt = mesolf_amd.summary_image_pixelwise(m, h, w, w1, w2, 3, 3)
    ri, rs, rt = O.summary_pixelwise(m, w1, w2, 3, 3)
    assert rel_l2(bs.ravel(order="F"), rs) <= 1e-9 and rel_l2(bt.ravel(), rt) <= 1e-9
    got, ok = img.ravel(order="F"), np.isfinite(ri)
    assert np.array_equal(np.isnan(got[~ok]), np.isnan(ri[~ok]))
    if T > 8:
        assert np.linalg.norm((got - ri)[ok]) <= 1e-5 * np.linalg.norm(ri[ok])


@pytest.mark.parametrize("h,w,T", EDGES)
def test_global(h, w, T):
    m = _movie(h * w, T)
    img, bs, bt = mesolf_amd.summary_image_global(m, h, w, 3)
    ri, rs, rt = O.summary_global(m, 3)
    assert rel_l2(bs.ravel(order="F"), rs) <= 1e-9 and rel_l2(bt.ravel(), rt) <= 1e-9
    if T > 8:
        ok = np.isfinite(ri)
        assert rel_l2(img.ravel(order="F")[ok], ri[ok]) <= 1e-5
