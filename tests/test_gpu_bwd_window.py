"""The backprojection's LDS ratio window at the edges of its tiles and at the
largest radii, against the FP64 oracle.

One view step with taps and an image of a few large values, so that a wrong
window cell shows.  Tolerance: the forward product (volume and taps) and the
backprojection (ratio and taps) round four operands to the precision's unit u
(2^-8 BF16, 2^-11 FP16; FP32 sums are far below), the normaliser's taps and the
volume's upper half two more: at most 6 u of the corrected volume.  FP32:
5e-6, as for the split view step.
"""
import numpy as np
import pytest

import mesolf_amd
from oracle import mesolf_oracle as O

pytestmark = pytest.mark.gpu

TOL = {"bf16": 6 * 2.0**-8, "fp16": 6 * 2.0**-11, "fp32": 5e-6}


@pytest.fixture(scope="module")
def ctx():
    c = mesolf_amd.Context(0)
    yield c
    c.close()


def _problem(ctx, rb):
    rng = np.random.default_rng(sum(rb))
    rf = [0] * len(rb)
    fwd = [0.5 + rng.random((1, 1, 15, 15)).astype(np.float32) for _ in rf]
    bwd = [(0.01 + rng.random((2 * r + 1, 2 * r + 1, 15, 15)) ** 8).astype(np.float32) for r in rb]
    cp = O.CompactPSF(N=15, Z=len(rb), views=[(7, 7)], weights=[0.3], rf=rf, rb=list(rb))
    cp.fwd.append([t.astype(np.float64) for t in fwd])
    cp.bwd.append([t.astype(np.float64) for t in bwd])
    psf = mesolf_amd.PSF.from_compact(
        ctx, cp.views, cp.weights, rf, np.concatenate([mesolf_amd.compact_block_layout(t) for t in fwd]), rb=rb,
        bwd_flat=np.concatenate([mesolf_amd.compact_block_layout(t) for t in bwd]))
    return cp, psf, rng


# 16 + 2 r window columns around whole 8-dword and 16-lenslet blocks, K-steps of one to many
@pytest.mark.parametrize("prec,rb,n1,n2", [
    ("bf16", (0, 1, 3), 1, 1), ("bf16", (4, 5), 17, 16), ("bf16", (13, 14), 33, 15), ("bf16", (37, 0), 40, 18),
    ("fp16", (0, 3, 4), 16, 33), ("fp16", (12, 20), 7, 31), ("fp16", (0, 37), 49, 5),
    ("fp32", (65, 2), 9, 20), ("fp32", (67,), 71, 3)])
def test_view_step_against_the_oracle(ctx, prec, rb, n1, n2):
    cp, psf, rng = _problem(ctx, rb)
    p = mesolf_amd.Patch(psf, n1, n2, prec)
    X = (0.1 + rng.random(p.shape)).astype(np.float32)
    LF = (1 + 200 * (rng.random(p.shape[:2]) < 0.1)).astype(np.float32)
    p.set_volume(X)
    p.set_image(LF)
    p.run(1, views_limit=1, filter=False)
    X = X.astype(np.float64)
    ref = O.rl_compact(LF.astype(np.float64), cp, 1, X0=X, views_limit=1, filter_planes=False)
    assert np.linalg.norm(p.get_volume() - ref) <= TOL[prec] * np.linalg.norm(ref - 0.7 * X)


@pytest.mark.parametrize("prec,r", [("bf16", 38), ("fp16", 38), ("fp32", 68)])
def test_larger_radii_are_refused(ctx, prec, r):
    _, psf, _ = _problem(ctx, (r,))
    with pytest.raises(mesolf_amd.MesolfError, match="too large"):
        mesolf_amd.Patch(psf, 4, 4, prec)
