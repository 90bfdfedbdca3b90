"""The FP32 view step on the BF16 matrix pipe (operands split into three BF16
parts) at the edges of its tiles, against the FP64 oracle.

Tolerance: a product leaves out three partial products of at most 2^-24 of it
each, and the FP32 sums (at most 48 steps of 24 matrix instructions, then the
planes) are rounded to 2^-24 of the partial sum a few hundred times with random
signs: below 20 * 2^-24 = 1.2e-6 of the summed sizes.  2e-6 is asked for, of a
view step 5e-6 (projection, ratio, backprojection, normaliser, product).
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O

pytestmark = pytest.mark.gpu


def _psf(radii, seed, low=0.05, views=((7, 7), (3, 9))):
    rng = np.random.default_rng(seed)
    cp = O.CompactPSF(N=15, Z=len(radii), views=list(views), weights=[0.3] * len(views), rf=list(radii),
                      rb=list(radii))
    flat = []
    for _ in views:
        fz = [(low + rng.random((2 * r + 1, 2 * r + 1, 15, 15))).astype(np.float32) for r in radii]
        flat += [mesolf_amd.compact_block_layout(t) for t in fz]
        cp.fwd.append([t.astype(np.float64) for t in fz])
        cp.bwd.append([np.ascontiguousarray(t[::-1, ::-1]).astype(np.float64) for t in fz])
    return cp, np.concatenate(flat)


def _patch(ctx, cp, flat, n1, n2):
    psf = mesolf_amd.PSF.from_compact(ctx, cp.views, cp.weights, cp.rf, flat)
    return mesolf_amd.Patch(psf, n1, n2, "fp32")


# radii around whole 16-tap tiles and 8-tap pieces (2 r + 1 = 15, 17, 31, 33, 47)
# and planes of one tap; grids below, at and past 16-lenslet and 8-column blocks
CASES = [((0, 1, 2), 1, 1), ((7, 8), 15, 9), ((15, 16), 17, 8), ((23, 3), 16, 16), ((23, 0), 33, 7),
         ((4, 12, 5), 50, 31), ((2, 3, 2), 5, 67)]


@pytest.fixture(scope="module")
def ctx():
    c = mesolf_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("radii,n1,n2", CASES)
def test_forward_and_view_step_against_the_oracle(ctx, radii, n1, n2):
    cp, flat = _psf(radii, seed=sum(radii) + n1)
    p = _patch(ctx, cp, flat, n1, n2)
    rng = np.random.default_rng(9)
    X = (rng.random(p.shape) ** 4).astype(np.float32)
    p.set_volume(X)
    Xl = O.to_lenslet(X.astype(np.float64), 15)
    for k in range(2):
        ref = O.forward_compact(Xl, cp.fwd[k], cp.rf)
        got = p.forward_view(k)
        assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)
    LF = rng.poisson(50.0, p.shape[:2]).astype(np.float32)
    p.set_image(LF)
    p.run(1, views_limit=2, filter=False)
    ref = O.rl_compact(LF.astype(np.float64), cp, 1, X0=X.astype(np.float64), views_limit=2, filter_planes=False)
    assert np.linalg.norm(p.get_volume() - ref) <= 5e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("value", [np.inf, np.nan, np.finfo(np.float32).max])
def test_volume_values_that_bf16_cannot_hold(ctx, value):
    """Infinities stay infinities, NaN stays NaN and FLT_MAX is summed like any
    other value, in the lenslets that the voxel reaches and nowhere else."""
    n1, n2 = 21, 12
    cp, flat = _psf((2, 9), seed=4)
    p = _patch(ctx, cp, flat, n1, n2)
    X = np.full(p.shape, 0.5, np.float32)
    X[15 * 10 + 3, 15 * 6 + 2, 0] = value
    p.set_volume(X)
    with np.errstate(all="ignore"):
        ref = O.forward_compact(O.to_lenslet(X.astype(np.float64), 15), cp.fwd[1], cp.rf).astype(np.float32)
    got = p.forward_view(1)
    reach = np.zeros((n1, n2), bool)
    reach[8:13, 4:9] = True
    if np.isfinite(value):
        assert np.array_equal(np.isfinite(got), np.isfinite(ref))
        m = np.isfinite(ref)
        assert np.allclose(got[m], ref[m], rtol=2e-6)
    else:
        assert np.isfinite(got[~reach]).all() and np.allclose(got[~reach], ref[~reach], rtol=2e-6)
        assert (np.isnan(got[reach]) if np.isnan(value) else got[reach] == np.inf).all()


def test_infinite_tap(ctx):
    cp, flat = _psf((1,), seed=2)
    flat = flat.copy()
    flat[(1 * 3 + 1) * 225 + 7 * 15 + 4] = np.inf  # view 0, centre offset, phase (4, 7)
    p = _patch(ctx, cp, flat, 6, 5)
    p.set_volume(np.ones(p.shape, np.float32))
    assert (p.forward_view(0) == np.inf).all() and np.isfinite(p.forward_view(1)).all()
