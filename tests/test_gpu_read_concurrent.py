"""Reading a large volume while other threads keep the context's stream busy."""
import threading
import time

import numpy as np
import pytest

import mesolf_amd

pytestmark = pytest.mark.gpu

Z = 11


@pytest.fixture(scope="module")
def ctx():
    c = mesolf_amd.Context(0)
    yield c
    c.close()


def _psf(ctx, radius, views, weight):
    rng = np.random.default_rng(3)
    K = 2 * radius + 1
    blocks = [(0.1 + rng.random((K, K, 15, 15))).astype(np.float32) for _ in range(Z)]
    one = np.concatenate([mesolf_amd.compact_block_layout(t) for t in blocks])
    return mesolf_amd.PSF.from_compact(ctx, views, [weight] * len(views), [radius] * Z, np.concatenate([one] * len(views)))


def test_a_read_does_not_wait_for_work_that_comes_after_it(ctx):
    """A read that begins behind a short piece of work ends long before a long one
    that another thread enqueues next."""
    psf = _psf(ctx, 8, [(u, v) for u in range(15) for v in range(15)][:60], 0.3)
    rng = np.random.default_rng(4)
    a, b = mesolf_amd.Patch(psf, 60, 60, "fp32"), mesolf_amd.Patch(psf, 90, 90, "fp32")
    for p in (a, b):
        p.set_image(rng.poisson(50.0, p.shape[:2]).astype(np.float32))
        p.init_volume()
    X = rng.random(b.shape).astype(np.float32)
    b.set_volume(X)
    assert np.array_equal(b.get_volume(f64=True), X)  # 160 MB; its buffers are made
    a.run(4)
    ctx.synchronize()
    got, took = [], []

    def read():
        t0 = time.perf_counter()
        got.append(b.get_volume(f64=True))
        took.append(time.perf_counter() - t0)

    a.run(20)  # the read waits for this
    th = threading.Thread(target=read)
    th.start()
    time.sleep(0.02)
    t0 = time.perf_counter()
    a.run(150)
    ctx.synchronize()
    work = time.perf_counter() - t0
    th.join()
    assert np.array_equal(got[0], X)
    assert took[0] < 0.5 * work, (took, work)


def test_a_volume_read_beside_its_batch_is_one_state(ctx):
    """All lenslets of the volume are alike in every state, so a volume put
    together from several would show."""
    psf = _psf(ctx, 0, [(7, 7)], 0.01)
    p = mesolf_amd.Patch(psf, 90, 90, "fp32")
    batch = mesolf_amd.Batch(psf, 1, "fp32")
    rng = np.random.default_rng(5)
    p.set_image(np.tile(rng.poisson(5000.0, (15, 15)).astype(np.float32), (90, 90)))
    X = np.tile(rng.random((15, 15, Z)).astype(np.float32), (90, 90, 1))
    p.set_volume(X)
    batch.attach(p)
    batch.run(1, False)
    p.get_volume(f64=True)
    stop = threading.Event()

    def work():
        while not stop.is_set():
            batch.run(1, False)

    for _ in range(3):
        p.set_volume(X)
        stop.clear()
        th = threading.Thread(target=work)
        th.start()
        time.sleep(0.01)
        v = p.get_volume(f64=True)
        stop.set()
        th.join()
        ctx.synchronize()
        assert not np.array_equal(v, X)
        t = v.reshape(90, 15, 90, 15, Z)
        assert (t == t[:1, :, :1]).all()
    batch.close()
