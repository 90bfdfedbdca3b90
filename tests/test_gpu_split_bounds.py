"""How far down the split of FP32 operands into three BF16 parts reaches.

The third part of a value ends at BF16's last bit, 2^-133, so values from 2^-110 keep
their 24 bits and smaller ones are up to 2^-134 off.  Inputs scaled by a power of two
down to 2^-110 give the same significands, and below that the error is what those
operand errors and the FP32 sums allow.
"""
import numpy as np
import pytest

import mesolf_amd
from mesolf_amd import synth
from tests.helpers import synthetic_problem

pytestmark = pytest.mark.gpu


def _half_to_one(shape, seed):
    return (0.5 + 0.5 * np.random.default_rng(seed).random(shape)).astype(np.float32)


@pytest.mark.parametrize("which", ["bitmap", "kernel"])
def test_mex_operands(which):
    """A sum of 961 terms is rounded 6 * 961 / 32 = 180 times per side, at most
    2 * sqrt(180) * 2^-24 = 1.6e-6 apart for roundings of random sign."""
    W, H, n, kw = 47, 33, 2, 31
    b, K = _half_to_one((W, H, n), 1), _half_to_one((kw, kw, 15, 15), 2)
    ref = mesolf_amd.mex_lfm_convolution_vec(b, K)
    for e in (-60, -90, -100, -109, -110, -112, -116, -120, -126):
        s = [a if w != which else np.ldexp(a, e).astype(np.float32) for w, a in (("bitmap", b), ("kernel", K))]
        got = mesolf_amd.mex_lfm_convolution_vec(*s)
        want = np.ldexp(ref.astype(np.float64), e)
        if e >= -109:  # values of 2^-110 and more
            assert np.array_equal(got, want.astype(np.float32)), e
        else:
            assert (np.abs(got - want) <= kw * kw * 2.0 ** -134 + 1.6e-6 * want).all(), e


def test_forward_projection():
    """Taps of at most t: the products end at FP32's last bit, 2^-149, like any
    FP32 sum; together with 2^-134 t per operand that bounds the error."""
    wl = synth.TINY
    tabs, cp, truth, LF = synthetic_problem(wl, seed=2)
    fwd = np.asarray(tabs["fwd"])
    t = float(np.abs(fwd).max())
    terms = 225 * sum((2 * r + 1) ** 2 for r in tabs["rf"])
    with mesolf_amd.Context(0) as ctx:
        psf = mesolf_amd.PSF.from_compact(ctx, tabs["uv"], tabs["weights"], tabs["rf"], tabs["fwd"])
        p = mesolf_amd.Patch(psf, wl.n1, wl.n2, "fp32")
        X = _half_to_one(p.shape, 3)
        p.set_volume(X)
        ref = p.project_all().astype(np.float64)
        for e in (-60, -90, -100, -110, -116, -120):
            p.set_volume(np.ldexp(X, e).astype(np.float32))
            got, want = p.project_all(), np.ldexp(ref, e)
            if e >= -90:  # nothing below the smallest normal number
                assert np.array_equal(got, want.astype(np.float32)), e
            else:
                assert (np.abs(got - want) <= terms * (2.0 ** -134 * t + 2.0 ** -149)
                        + 2e-6 * want).all(), e
        p.close()
        psf.close()
