"""A bitmap's MEX result does not depend on the call it is part of: bit for bit the
same alone, among any number of others (which changes the workgroups' shape), and
summed in a segment call.
"""
import numpy as np
import pytest

import mesolf_amd

pytestmark = pytest.mark.gpu


def _inputs(W, H, n, kw, seed=17):
    rng = np.random.default_rng(seed)
    return (rng.random((W, H, n)).astype(np.float32), (rng.random((kw, kw, 15, 15)) - 0.2).astype(np.float32))


# small bitmaps of few row groups to wide ones of many; kernels of one K-step to
# many, narrower and wider than the bitmap, fewer and more rows than classes
@pytest.mark.parametrize("W,H,kw,counts", [
    (47, 33, 31, (1, 2, 3, 5, 9, 17, 33, 65, 160)), (150, 137, 61, (1, 2, 4, 8, 16, 48, 96)),
    (16, 5, 5, (1, 7, 60, 300)), (90, 7, 241, (1, 3, 20, 90)), (396, 110, 121, (1, 2, 4, 9, 24, 50)),
    (31, 200, 7, (1, 4, 30, 120)), (225, 60, 13, (1, 8, 64)),
    # many rows and several lengths of batch: the shapes of three and four rows to a
    # workgroup, and those of many cells, each against one bitmap's small shape
    (130, 513, 61, (1, 4, 8, 16, 30, 60)), (130, 513, 17, (1, 8, 16, 30, 60)), (77, 1501, 33, (1, 16, 30)),
    (640, 9, 5, (1, 24, 48)),
])
def test_any_number_of_bitmaps(W, H, kw, counts):
    b, K = _inputs(W, H, counts[-1], kw)
    whole = mesolf_amd.mex_lfm_convolution_vec(b, K)
    for n in counts[:-1]:
        got = mesolf_amd.mex_lfm_convolution_vec(b[:, :, -n:], K)
        assert np.array_equal(got, whole[:, :, -n:]), (n, float(np.abs(got - whole[:, :, -n:]).max()))


@pytest.mark.parametrize("W,H,kw,nseg", [(47, 33, 31, 3), (150, 137, 61, 12), (61, 40, 5, 40), (396, 50, 91, 30)])
def test_segments_are_sums_of_calls(W, H, kw, nseg):
    """Planes repeated within a segment and missing from others, added in plane
    order, slices of a plane in slice order."""
    rng = np.random.default_rng(nseg)
    Z = 3
    ptr = np.concatenate([[0], np.cumsum(rng.integers(1, 5, nseg))]).astype(np.int64)
    plane = rng.integers(0, Z, ptr[-1]).astype(np.int32)
    b = rng.random((W, H, len(plane))).astype(np.float32)
    K = np.asfortranarray((rng.random((kw, kw, 15, 15, Z)) - 0.2).astype(np.float32))
    got = mesolf_amd.lfm_convolution_segments(b, plane, ptr, K)
    for s in {0, nseg // 2, nseg - 1}:
        want = np.zeros((W, H), np.float32)
        for i in sorted(range(ptr[s], ptr[s + 1]), key=lambda i: plane[i]):
            want = want + mesolf_amd.mex_lfm_convolution_vec(b[:, :, i:i + 1], K[..., plane[i]])[:, :, 0]
        assert np.array_equal(got[:, :, s], want), s
