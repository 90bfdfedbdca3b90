"""Reading volumes back below and above the size from which several threads
copy them out (64 MiB, chunks of 4 MiB): the values that were set, exactly."""
import threading

import numpy as np
import pytest

import mesolf_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def psf():
    ctx = mesolf_amd.Context(0)
    block = mesolf_amd.compact_block_layout(np.ones((1, 1, 15, 15), np.float32))
    psf = mesolf_amd.PSF.from_compact(ctx, [(7, 7)], [0.3], [0, 0, 0], np.concatenate([block] * 3))
    yield psf
    psf.close()
    ctx.close()


# float32 MiB: 0.03, 32.006, 31.996 (their float64: just above, with a last chunk of few
# elements, and just below the line) and 65.9
@pytest.mark.parametrize("n1,n2", [(3, 4), (113, 110), (109, 114), (160, 160)])
def test_set_and_read_back(psf, n1, n2):
    p = mesolf_amd.Patch(psf, n1, n2, "fp32")
    X = np.random.default_rng(n1).random(p.shape).astype(np.float32)
    p.set_volume(X)
    assert np.array_equal(p.get_volume(), X)
    assert np.array_equal(p.get_volume(f64=True), X.astype(np.float64))
    p.close()


def test_two_threads_read_at_once(psf):
    patches = [mesolf_amd.Patch(psf, 170, 160 + k, "fp32") for k in range(2)]
    want = [np.random.default_rng(k).random(p.shape).astype(np.float32) for k, p in enumerate(patches)]
    for p, x in zip(patches, want):
        p.set_volume(x)
    got = [None, None]

    def read(k):
        got[k] = [patches[k].get_volume() for _ in range(3)]

    threads = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert all(np.array_equal(g, want[k]) for g in got[k])
        patches[k].close()
