"""Which bitmaps of a MEX call go to the FP32 form (mex_marks.h).

A value that the split form cannot hold sends its own bitmap there, or, in a
kernel set, the slices on that set; every other bitmap keeps the bits that it has
in a call without such values, and so do later calls.  All comparisons are bit
for bit.
"""
import ctypes as C

import numpy as np
import pytest

import mesolf_amd
from mesolf_amd import lib as L

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    c = mesolf_amd.Context(0)
    yield c
    c.close()


def _inputs(W, H, n, kw, seed=11):
    rng = np.random.default_rng(seed)
    return (rng.random((W, H, n)).astype(np.float32), (rng.random((kw, kw, 15, 15)) - 0.2).astype(np.float32))


def _equal(a, b):
    return np.array_equal(a, b, equal_nan=True)


# marked bitmaps first, last and between; more bitmaps than one block's; one-pixel bitmaps
@pytest.mark.parametrize("W,H,n,kw,bad", [(47, 33, 5, 31, [2]), (46, 20, 40, 17, [0, 21, 39]), (150, 60, 3, 61, [1, 2]),
                                          (1, 1, 200, 5, [77]), (2, 3, 5000, 5, [4500])])
@pytest.mark.parametrize("value", [np.inf, np.nan, np.finfo(np.float32).max])
def test_a_marked_bitmap_leaves_the_others(W, H, n, kw, bad, value):
    b, K = _inputs(W, H, n, kw)
    clean = mesolf_amd.mex_lfm_convolution_vec(b, K)
    b2 = b.copy()
    b2[W // 2, H // 2, bad] = value
    got = mesolf_amd.mex_lfm_convolution_vec(b2, K)
    rest = np.setdiff1d(np.arange(n), bad)
    assert _equal(got[:, :, rest], clean[:, :, rest])
    for i in bad[:1]:
        assert _equal(got[:, :, i:i + 1], mesolf_amd.mex_lfm_convolution_vec(b2[:, :, i:i + 1], K))
        assert not _equal(got[:, :, i], clean[:, :, i])


def test_a_marked_kernel_set_takes_its_own_slices():
    W, H, kw, Z = 60, 31, 31, 3
    plane = np.array([0, 2, 1, 0, 1, 2, 0, 2], np.int32)
    ptr = np.array([0, 2, 3, 5, 6, 8], np.int64)  # the first, fourth and fifth segments stay off plane 1
    b, _ = _inputs(W, H, len(plane), kw)
    rng = np.random.default_rng(5)
    K = np.asfortranarray((rng.random((kw, kw, 15, 15, Z)) - 0.2).astype(np.float32))
    clean = mesolf_amd.lfm_convolution_segments(b, plane, ptr, K)
    K2 = K.copy(order="F")
    K2[3, 4, 5, 6, 1] = np.inf
    got = mesolf_amd.lfm_convolution_segments(b, plane, ptr, K2)
    assert _equal(got[:, :, [0, 3, 4]], clean[:, :, [0, 3, 4]])
    assert not np.isfinite(got[:, :, 1]).all() and not np.isfinite(got[:, :, 2]).all()
    b2 = b.copy()
    b2[20, 10, 3] = np.nan  # third segment
    got = mesolf_amd.lfm_convolution_segments(b2, plane, ptr, K)
    assert _equal(got[:, :, [0, 1, 3, 4]], clean[:, :, [0, 1, 3, 4]]) and np.isnan(got[20, 10, 2])
    assert _equal(mesolf_amd.lfm_convolution_segments(b, plane, ptr, K), clean)


@pytest.mark.parametrize("entry", ["mlf_lfm_convolution_vec_device", "mlf_lfm_convolution_vec_noalloc"])
def test_marks_end_with_their_call(ctx, entry):
    lib = L.load_library()
    W, H, n, kw = 61, 34, 3, 31
    b, K = _inputs(W, H, n, kw)
    bad = b.copy()
    bad[30, 20, 1] = np.inf
    Kbad = K.copy()
    Kbad[1, 2, 3, 4] = np.nan
    dev = [torch.from_numpy(a.ravel(order="F").copy()).to("cuda:0") for a in (b, bad, K, Kbad)]
    out = torch.empty(W * H * n, device="cuda:0")
    torch.cuda.synchronize()
    seen = []
    for im, k in ((0, 2), (1, 2), (0, 2), (0, 3), (1, 3), (0, 2)):
        L._check(getattr(lib, entry)(ctx.handle, C.c_void_p(dev[im].data_ptr()), W, H, n,
                                     C.c_void_p(dev[k].data_ptr()), kw, 15, C.c_void_p(out.data_ptr())))
        ctx.synchronize()
        seen.append(out.cpu().numpy())
    assert np.isfinite(seen[0]).all() and not np.isfinite(seen[1]).all() and np.isnan(seen[3]).any()
    assert _equal(seen[2], seen[0]) and _equal(seen[5], seen[0])
