"""The depth filter on axes of two and four lenslets, whose even period is too short
for the ends of the kernel to vanish: its middle tap counts.

The filter alone, against the oracle's FFT form: each pass sums at most 60 taps in
FP32, below 60 * 2^-24 = 3.6e-6 of the summed sizes, and the scale restores the
planes' sums to 1e-6: 8.2e-6.
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = mesolf_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n1,n2", [(2, 1), (1, 2), (2, 2), (4, 2), (2, 9), (4, 4), (3, 2), (6, 4)])
def test_filter(ctx, n1, n2):
    Z = 11
    rng = np.random.default_rng(n1 + 10 * n2)
    one = mesolf_amd.compact_block_layout(np.ones((1, 1, 15, 15), np.float32))
    psf = mesolf_amd.PSF.from_compact(ctx, [(7, 7)], [0.3], [0] * Z, np.concatenate([one] * Z))
    p = mesolf_amd.Patch(psf, n1, n2, "fp32")
    X = rng.random(p.shape).astype(np.float32)
    p.set_volume(X)
    p.sample_filter()
    ref = O.sample_filter_literal(X.astype(np.float64), O.filter_bank(*X.shape[:2], Z, 15))
    assert np.linalg.norm(p.get_volume() - ref) <= 8.2e-6 * np.linalg.norm(ref)
