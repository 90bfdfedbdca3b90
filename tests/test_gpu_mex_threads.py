"""MEX calls of several threads on one context: each call's launches share a scratch and
follow one another on the stream, so every result is that of the call alone."""
import ctypes as C
import threading

import numpy as np
import pytest

import mesolf_amd
from mesolf_amd import lib as L

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("entry", ["mlf_lfm_convolution_vec_device", "mlf_lfm_convolution_vec_noalloc"])
def test_threads_on_one_context(entry):
    lib = L.load_library()
    ctx = mesolf_amd.Context(0)
    W, H, kw = 61, 34, 31
    rng = np.random.default_rng(9)

    def dev(a):
        return torch.from_numpy(a.ravel(order="F").copy()).to("cuda:0")

    jobs = []
    for t in range(4):
        n = t + 1
        b = rng.random((W, H, n)).astype(np.float32)
        K = (rng.random((kw, kw, 15, 15)) - 0.2).astype(np.float32)
        if t == 3:
            b[5, 5, 1] = np.inf  # a call with a marked bitmap among the others
        jobs.append((dev(b), n, dev(K), [torch.empty(W * H * n, device="cuda:0") for _ in range(60)]))
    torch.cuda.synchronize()

    def call(job, out):
        L._check(getattr(lib, entry)(ctx.handle, C.c_void_p(job[0].data_ptr()), W, H, job[1],
                                     C.c_void_p(job[2].data_ptr()), kw, 15, C.c_void_p(out.data_ptr())))

    want = []
    for job in jobs:
        call(job, job[3][0])
        ctx.synchronize()
        want.append(job[3][0].clone())
    threads = [threading.Thread(target=lambda job=job: [call(job, o) for o in job[3]]) for job in jobs]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    ctx.synchronize()
    for job, w in zip(jobs, want):
        for o in job[3]:
            assert torch.equal(torch.nan_to_num(o), torch.nan_to_num(w))
    ctx.close()
