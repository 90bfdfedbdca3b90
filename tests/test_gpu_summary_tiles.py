"""The tile passes of the summary image at the edges of their ranges: tiles of
64, 32 and 16 pixels, their frame limits, the longer movies that go without
tiles, ragged pixel counts, windows past the movie's length (not a smoothing window
over the whole movie: the smoothed movie is then constant and the image is the
sign of a rounding error).

Tolerances: backgrounds are FP64 sums of at most 1e6 terms in another order,
1e-9 of the result; the detrended movie is rounded to FP32 (2^-24) before a
smoothing, a third power and a standard deviation that loses at most two
decimal digits here: 1e-5.
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


def _movie(npix, T, seed=1):
    rng = np.random.default_rng(seed)
    base = 200 + 50 * rng.random((npix, 1))
    return np.asfortranarray(rng.poisson(base * (1 + 0.3 * np.sin(np.arange(T) / 7.0))).astype(np.float32))


@pytest.mark.parametrize("h,w,T,w1,w2", [
    (1, 1, 2, 3, 1), (7, 9, 1, 1, 1), (5, 13, 8, 20, 8), (33, 31, 250, 100, 20), (10, 13, 500, 99, 3),
    (9, 7, 512, 100, 21), (6, 11, 590, 40, 20), (5, 8, 700, 150, 30), (4, 9, 960, 101, 20), (3, 7, 1000, 100, 20),
    (21, 5, 1200, 64, 7),
])
def test_pixelwise_against_the_oracle(h, w, T, w1, w2):
    m = _movie(h * w, T)
    img, bs, bt = mesolf_amd.summary_image_pixelwise(m, h, w, w1, w2, 3, 3)
    ri, rs, rt = O.summary_pixelwise(m, w1, w2, 3, 3)
    assert rel_l2(bs.ravel(order="F"), rs) <= 1e-9 and rel_l2(bt.ravel(), rt) <= 1e-9
    got, ref = img.ravel(order="F"), ri
    ok = np.isfinite(ref)
    assert np.array_equal(np.isnan(got[~ok]), np.isnan(ref[~ok]))
    if ok.any() and T > 8:
        assert np.linalg.norm((got - ref)[ok]) <= 1e-5 * np.linalg.norm(ref[ok])


@pytest.mark.parametrize("T,bg_iter", [(3, 1), (300, 5), (600, 2), (1100, 2)])
def test_global_against_the_oracle(T, bg_iter):
    h, w = 19, 23
    m = _movie(h * w, T, seed=4)
    img, bs, bt = mesolf_amd.summary_image_global(m, h, w, bg_iter)
    ri, rs, rt = O.summary_global(m, bg_iter)
    assert rel_l2(bs.ravel(order="F"), rs) <= 1e-9 and rel_l2(bt.ravel(), rt) <= 1e-9
    ok = np.isfinite(ri)
    assert rel_l2(img.ravel(order="F")[ok], ri[ok]) <= 1e-5


def test_nan_pixel_stays_in_its_pixel_and_zero_movie_is_nan():
    h, w, T = 16, 9, 130
    m = _movie(h * w, T)
    m[70, 40] = np.nan
    img, bs, bt = mesolf_amd.summary_image_pixelwise(m, h, w, 20, 5, 3, 1)
    img = img.ravel(order="F")
    assert np.isnan(img[70]) and np.isfinite(np.delete(img, 70)).all() and np.isnan(bt).any()
    z = mesolf_amd.summary_image_pixelwise(np.zeros((h * w, T), np.float32), h, w, 20, 5, 3, 2)
    assert all(np.isnan(a).all() for a in z)
