"""Workloads that the performance of this framework is measured on.

Each case is one call sequence of a user's program: a whole reconstruction of a
patch (the headline patch, a carpet patch, the small patch through the MATLAB
drop-in), a serving batch, the forward projection of a volume, the MEX operator
and the seed-library loop on it, the summary image and the rectification of a
recording.  `listed` names them, `draw` gives more of the same ranges.

The optical system is one for the whole file, as a microscope has one: 15
phases per lenslet, 177 views in the aperture, Gaussian view kernels that widen
and shift with depth (radius 2 lenslets in focus, 17 at 100 um), kept resident
like a program keeps it.  Images, volumes, movies and bitmaps come from the
seed.
"""
from __future__ import annotations

import ctypes
import functools
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import mesolf_amd

N = 15          # phases per lenslet axis
C = 7           # centre phase
NP = N * N
VOLUME_CACHE = 256 << 20  # bytes the last-level cache holds


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # the headline patch: 101 x 101 lenslets, 51 planes, 8 iterations, BF16
        {"name": "rl_bf16_101x101x51", "kind": "rl", "prec": "bf16", "n1": 101, "n2": 101, "planes": 51,
         "iters": 8},
        # a carpet patch of a recording (ragged sides, 3 iterations as the demo
        # runs it) at the default precision
        {"name": "rl_fp32_61x67x51", "kind": "rl", "prec": "fp32", "n1": 61, "n2": 67, "planes": 51, "iters": 3},
        # the same at FP16, fewer planes
        {"name": "rl_fp16_81x73x31", "kind": "rl", "prec": "fp16", "n1": 81, "n2": 73, "planes": 31, "iters": 3},
        # a small region of interest: few workgroups per launch, 1416 dependent view steps
        {"name": "rl_bf16_33x33x11", "kind": "rl", "prec": "bf16", "n1": 33, "n2": 33, "planes": 11, "iters": 8},
        # the drop-in for the MATLAB function with dense PSFs on the host
        {"name": "recon_fp32_33x33x11", "kind": "recon", "prec": "fp32", "n1": 33, "n2": 33, "planes": 11,
         "iters": 8},
        # serving: uneven patches of one recording in shared launches
        {"name": "batch_bf16_3x45to75x51", "kind": "batch", "prec": "bf16", "grids": "45x52,61x58,75x75",
         "planes": 51, "iters": 3},
        # the forward direction alone: sensor image of a volume, all views
        {"name": "project_fp32_81x81x51", "kind": "project", "prec": "fp32", "n1": 81, "n2": 81, "planes": 51},
        # the MEX operator at the demo's bitmap and kernel size
        {"name": "mex_396x396x96_kw241", "kind": "mex", "w": 396, "h": 396, "n": 96, "kw": 241},
        # ... and its smallest call: one small bitmap, an in-focus kernel
        {"name": "mex_150x137x1_kw61", "kind": "mex", "w": 150, "h": 137, "n": 1, "kw": 61},
        # the seed library: slices of many segments over several planes
        {"name": "seedlib_396x396_24seg_5z", "kind": "seedlib", "w": 396, "h": 396, "segments": 24, "z": 5,
         "kw": 241},
        # the summary image and rank-1 background of a carpet patch's movie
        {"name": "summary_765x750x400", "kind": "summary", "h": 765, "w": 750, "t": 400, "w1": 100, "w2": 20,
         "mode": "pixelwise"},
        # rectification of raw frames (14.8-px lenslet pitch)
        {"name": "rectify_1515x1515x64", "kind": "rectify", "h": 1515, "w": 1515, "t": 64, "dx": 14.8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["rl", "rl", "rl", "recon", "batch", "project", "mex", "mex", "seedlib", "summary",
                           "summary", "rectify"])
        if kind == "rl":
            c = {"kind": kind, "prec": rng.choice(["fp32", "bf16", "bf16", "fp16"]), "n1": _log_int(rng, 20, 101),
                 "n2": _log_int(rng, 20, 101), "planes": _log_int(rng, 7, 51), "iters": rng.randint(1, 8)}
            cost = work(c)["flops"] * (6 if c["prec"] == "fp32" else 1.5)
        elif kind == "recon":
            c = {"kind": kind, "prec": rng.choice(["fp32", "fp32", "bf16"]), "n1": rng.randint(12, 40),
                 "n2": rng.randint(12, 40), "planes": rng.randint(3, 11), "iters": rng.randint(1, 8)}
            cost = work(c)["flops"] * 6
        elif kind == "batch":
            g = ",".join("%dx%d" % (rng.randint(30, 80), rng.randint(30, 80)) for _ in range(rng.randint(2, 5)))
            c = {"kind": kind, "prec": rng.choice(["bf16", "bf16", "fp32"]), "grids": g,
                 "planes": _log_int(rng, 11, 51), "iters": rng.randint(1, 3)}
            cost = work(c)["flops"] * (6 if c["prec"] == "fp32" else 1.5)
        elif kind == "project":
            c = {"kind": kind, "prec": rng.choice(["fp32", "bf16", "fp16"]), "n1": _log_int(rng, 16, 101),
                 "n2": _log_int(rng, 16, 101), "planes": _log_int(rng, 5, 51)}
            cost = work(c)["flops"] * 12
        elif kind == "mex":
            c = {"kind": kind, "w": _log_int(rng, 90, 500), "h": _log_int(rng, 90, 500), "n": _log_int(rng, 1, 128),
                 "kw": 2 * _log_int(rng, 15, 125) + 1}
            cost = work(c)["flops"] * 3
        elif kind == "seedlib":
            c = {"kind": kind, "w": rng.randint(200, 420), "h": rng.randint(200, 420),
                 "segments": rng.randint(2, 60), "z": rng.randint(1, 8), "kw": 2 * rng.randint(45, 120) + 1}
            cost = work(c)["flops"] * 3
        elif kind == "summary":
            c = {"kind": kind, "h": _log_int(rng, 100, 1000), "w": _log_int(rng, 100, 1000),
                 "t": _log_int(rng, 40, 800), "w1": rng.randint(20, 150), "w2": rng.randint(3, 30),
                 "mode": rng.choice(["pixelwise", "pixelwise", "global"])}
            cost = 0 if c["h"] * c["w"] * c["t"] < 4e8 else float("inf")
        else:
            c = {"kind": kind, "h": rng.randint(500, 2000), "w": rng.randint(500, 2000), "t": _log_int(rng, 4, 80),
                 "dx": round(rng.uniform(13.5, 16.5), 2)}
            cost = 0
        if cost <= most:
            return c


# ------------------------------------------------------------------ the optics
def _z_um(planes):
    return [4 * (i - planes // 2) for i in range(planes)]


def _radius(z):
    return (15 * abs(z) + 99) // 100 + 2


def _views():
    """Views of the aperture disc in the reconstruction's visiting order, a
    spiral from the rim inwards."""
    order, lo, hi = [], 0, N - 1
    while lo < hi:
        order += [(i, lo) for i in range(lo, hi + 1)] + [(hi, j) for j in range(lo + 1, hi + 1)]
        order += [(i, hi) for i in range(hi - 1, lo - 1, -1)] + [(lo, j) for j in range(hi - 1, lo, -1)]
        lo, hi = lo + 1, hi - 1
    order.append((C, C))
    return [(u, v) for u, v in order if (u - C) ** 2 + (v - C) ** 2 <= 7.5 ** 2]


def _factor(a, z):
    """[2r + 1, 15] factor of a view kernel along one axis: offset d, phase s."""
    r = _radius(z)
    x = N * np.arange(-r, r + 1)[:, None] + C - np.arange(N)[None, :]
    g = np.exp(-((x - N * 0.08 * z * (a - C) / 7.0) ** 2) / (2 * (15.0 * (1.0 + 0.1 * abs(z))) ** 2))
    g *= np.abs(x) <= N * r
    return g / g.sum() * N


@functools.lru_cache(maxsize=2)
def _tables(planes):
    """Forward tables of all views and planes, FP32, [d2, d1, s2, s1] blocks."""
    z_um, views = _z_um(planes), _views()
    blocks = [(2 * _radius(z) + 1) ** 2 * NP for z in z_um]
    out = np.empty(len(views) * sum(blocks), np.float32)

    def fill(k):
        u, v = views[k]
        o = k * sum(blocks)
        for z, n in zip(z_um, blocks):
            fx = _factor(u, z).astype(np.float32)
            fy = (_factor(v, z) / (len(views) * NP)).astype(np.float32)
            K = fx.shape[0]
            np.multiply(fy[:, None, :, None], fx[None, :, None, :], out=out[o:o + n].reshape(K, K, N, N))
            o += n

    with ThreadPoolExecutor(8) as ex:
        list(ex.map(fill, range(len(views))))
    return out


@functools.lru_cache(maxsize=1)
def _ctx():
    return mesolf_amd.Context(0)


@functools.lru_cache(maxsize=2)
def _psf(planes):
    views = _views()
    return mesolf_amd.PSF.from_compact(_ctx(), views, np.full(len(views), 0.3), [_radius(z) for z in _z_um(planes)],
                                       _tables(planes))


@functools.lru_cache(maxsize=1)
def _dense(planes):
    """Raw PSF pair H, Ht [S, S, 15, 15, planes] (single, column-major) whose
    phase-space tables are `_tables`, Ht the adjoint of H."""
    z_um, views, tabs = _z_um(planes), _views(), _tables(planes)
    R = max(_radius(z) for z in z_um)
    S = N * (2 * R + 1)
    H = np.zeros((S, S, N, N, planes), np.float32, order="F")
    Ht = np.zeros((S, S, N, N, planes), np.float32, order="F")
    s = np.arange(N)
    o = 0
    for u, v in views:
        for zi, z in enumerate(z_um):
            r = _radius(z)
            K = 2 * r + 1
            d = np.arange(-r, r + 1)
            t = tabs[o:o + K * K * NP].reshape(K, K, N, N).transpose(1, 0, 3, 2)  # [d1, d2, s1, s2]
            o += K * K * NP
            ok = np.abs(N * d[:, None] + C - s) <= N * r                          # the kernel's support
            d1, s1 = np.nonzero(ok)
            part = t[d1[:, None], d1[None, :], s1[:, None], s1[None, :]]
            xu, xv = u + N * (d[d1] + R) - s1 + C, v + N * (d[d1] + R) - s1 + C
            H[xu[:, None], xv[None, :], s1[:, None], s1[None, :], zi] = part
            xu, xv = N * (R - d[d1]) + C + s1 - u, N * (R - d[d1]) + C + s1 - v
            Ht[xu[:, None], xv[None, :], u, v, zi] = part
    return H, Ht


# ------------------------------------------------------------------ the inputs
def _spheres(rng, n1, n2, planes):
    n = max(2, n1 * n2 * 400 // 10201)
    return (rng.uniform(0, N * n1, n), rng.uniform(0, N * n2, n), rng.integers(0, planes, n),
            rng.uniform(0.5, 1.0, n))


def _image(rng, n1, n2, planes):
    """Sensor image of fluorescent cells over background, in photon counts."""
    cx, cy, zi, amp = _spheres(rng, n1, n2, planes)
    z = np.array(_z_um(planes), np.float64)[zi]
    s2 = 2 * (25.0 ** 2 + (15 + 1.5 * np.abs(z)) ** 2)

    def axis(n, c):
        u = np.arange(N * n) % N
        p = N * (np.arange(N * n) // N) + C
        return np.exp(-((p[:, None] - c - 1.2 * z * (u[:, None] - C) / 7.0) ** 2) / s2)

    clean = 0.05 + (axis(n1, cx) * amp) @ axis(n2, cy).T
    return np.asfortranarray(rng.poisson(clean * (1000.0 / clean.max())).astype(np.float32))


def _volume(rng, n1, n2, planes):
    """Cells (spheres of radius 3 lenslets and 3 planes) over background."""
    vol = np.full((N * n1, N * n2, planes), 0.01, np.float32, order="F")
    for x, y, z, a in zip(*_spheres(rng, n1, n2, planes)):
        x0, y0, z0 = max(0, int(x) - 45), max(0, int(y) - 45), max(0, int(z) - 3)
        box = vol[x0:int(x) + 46, y0:int(y) + 46, z0:int(z) + 4]
        gx, gy, gz = (np.arange(m) for m in box.shape)
        box += np.float32(a) * (((gx[:, None, None] + x0 - x) / 45) ** 2 + ((gy[None, :, None] + y0 - y) / 45) ** 2
                                + ((gz[None, None, :] + z0 - z) / 3.5) ** 2 <= 1)
    return vol


def _bitmaps(gen, w, h, n):
    """[n, h, w] slices of segments: one disc of fluorescence in each."""
    yy = torch.arange(h, device="cuda")[None, :, None]
    xx = torch.arange(w, device="cuda")[None, None, :]
    cx = torch.rand((n, 1, 1), device="cuda", generator=gen) * w
    cy = torch.rand((n, 1, 1), device="cuda", generator=gen) * h
    r = 8 + 30 * torch.rand((n, 1, 1), device="cuda", generator=gen)
    val = torch.rand((n, h, w), device="cuda", generator=gen)
    return (val * (((xx - cx) ** 2 + (yy - cy) ** 2) < r * r)).contiguous()


def _mex_kernels(gen, kw, z):
    """[z, 15, 15, kw, kw] kernels, each phase a speckled spot of unit sum."""
    d = torch.arange(kw, device="cuda") - kw // 2
    e = torch.stack([torch.exp(-((d - (s - C)) / (kw / 5.0)) ** 2) for s in range(N)])  # [15, kw]
    k = e[None, :, None, :, None] * e[None, None, :, None, :]
    k = k * (0.2 + torch.rand((z, N, N, kw, kw), device="cuda", generator=gen))
    return (k / k.sum(dim=(-1, -2), keepdim=True)).float().contiguous()


def _movie(gen, h, w, t):
    """[t, w, h] photon counts: vignetted background that bleaches, cells that flare."""
    y = torch.linspace(-1, 1, h, device="cuda")[None, :]
    x = torch.linspace(-1, 1, w, device="cuda")[:, None]
    j = torch.arange(t, device="cuda", dtype=torch.float32)
    base = 200 + 300 * torch.exp(-(x * x + y * y))
    cells = torch.rand((w, h), device="cuda", generator=gen) < 0.02
    rate = (0.85 + 0.15 * torch.exp(-j / (0.5 * t))) * (1 + 0.02 * torch.sin(j / 9.0))
    flare = (torch.rand((t,), device="cuda", generator=gen) < 0.05).float()
    out = torch.empty((t, w, h), device="cuda")
    for k in range(t):
        lam = base * rate[k] + 150.0 * flare[k] * cells
        out[k] = torch.poisson(lam, generator=gen)
    return out


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _grids(case):
    return [tuple(int(x) for x in g.split("x")) for g in case["grids"].split(",")]


def _segments(case, seed):
    """Planes of each segment's slices: a run of neighbouring planes."""
    rng = np.random.default_rng(seed)
    planes, ptr = [], [0]
    for _ in range(case["segments"]):
        a = int(rng.integers(0, case["z"]))
        planes += range(a, int(rng.integers(a, case["z"])) + 1)
        ptr.append(len(planes))
    return planes, ptr


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "kind": kind}
    rng = np.random.default_rng(seed)
    if kind == "rl":
        st["patch"] = mesolf_amd.Patch(_psf(case["planes"]), case["n1"], case["n2"], case["prec"])
        st["image"] = _image(rng, case["n1"], case["n2"], case["planes"])
    elif kind == "recon":
        st["H"], st["Ht"] = _dense(case["planes"])
        st["image"] = _image(rng, case["n1"], case["n2"], case["planes"])
    elif kind == "batch":
        psf = _psf(case["planes"])
        st["patches"] = [mesolf_amd.Patch(psf, a, b, case["prec"]) for a, b in _grids(case)]
        st["images"] = [_image(rng, a, b, case["planes"]) for a, b in _grids(case)]
        st["batch"] = mesolf_amd.Batch(psf, len(st["patches"]), case["prec"])
        for p in st["patches"]:
            st["batch"].attach(p)
    elif kind == "project":
        st["patch"] = mesolf_amd.Patch(_psf(case["planes"]), case["n1"], case["n2"], case["prec"])
        st["patch"].set_volume(_volume(rng, case["n1"], case["n2"], case["planes"]))
    elif kind == "mex":
        g = _gen(seed)
        st["bitmap"] = _bitmaps(g, case["w"], case["h"], case["n"])
        st["kernels"] = _mex_kernels(g, case["kw"], 1)
        st["out"] = torch.empty_like(st["bitmap"])
    elif kind == "seedlib":
        g = _gen(seed)
        st["planes"], st["ptr"] = _segments(case, seed)
        st["slices"] = _bitmaps(g, case["w"], case["h"], len(st["planes"]))
        st["kernels"] = _mex_kernels(g, case["kw"], case["z"])
        st["out"] = torch.empty((case["segments"], case["h"], case["w"]), device="cuda")
    elif kind == "summary":
        st["movie"] = _movie(_gen(seed), case["h"], case["w"], case["t"])
        st["out"] = {"image": torch.empty((case["w"], case["h"]), device="cuda", dtype=torch.float64),
                     "spatial": torch.empty((case["w"], case["h"]), device="cuda", dtype=torch.float64),
                     "temporal": torch.empty((case["t"],), device="cuda", dtype=torch.float64)}
    else:
        hq, wq = mesolf_amd.rectify_size(case["h"], case["w"], 8.3, 7.9, N, case["dx"])
        st["frames"] = _movie(_gen(seed), case["h"], case["w"], case["t"])
        st["out"] = torch.empty((case["t"], wq, hq), device="cuda")
    if kind in ("mex", "seedlib", "summary", "rectify"):
        torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return st


# ---------------------------------------------------------------- one pass
def _call(name, *args):
    """A device entry point of the C interface on the context's stream."""
    ctx = _ctx()
    lib = mesolf_amd.load_library()
    args = [ctypes.c_void_p(a.data_ptr()) if isinstance(a, torch.Tensor) else a for a in args]
    status = getattr(lib, name)(ctx.handle, *args)
    if status != 0:
        raise RuntimeError("%s: %s" % (name, lib.mlf_last_error().decode()))


def run(state):
    c, kind = state["case"], state["kind"]
    if kind == "rl":
        p = state["patch"]
        p.set_image(state["image"])
        p.init_volume()
        p.run(c["iters"])
        return p.get_volume()
    if kind == "recon":
        vol = mesolf_amd.recon_theory_phase_space_LFM_with_filter(
            state["image"], state["H"], state["Ht"], c["iters"], True, 1, precision=c["prec"])
        return vol.astype(np.float32)  # the drop-in's doubles hold single-precision values
    if kind == "batch":
        for p, im in zip(state["patches"], state["images"]):
            p.set_image(im)
            p.init_volume()
        state["batch"].run(c["iters"])
        return [p.get_volume() for p in state["patches"]]
    if kind == "project":
        return state["patch"].project_all()
    if kind == "mex":
        _call("mlf_lfm_convolution_vec_device", state["bitmap"], c["w"], c["h"], c["n"], state["kernels"], c["kw"],
              N, state["out"])
    elif kind == "seedlib":
        mesolf_amd.lfm_convolution_segments_device(
            _ctx(), state["slices"].data_ptr(), c["w"], c["h"], len(state["planes"]), state["planes"], state["ptr"],
            state["kernels"].data_ptr(), c["kw"], c["z"], state["out"].data_ptr())
    elif kind == "summary":
        o = state["out"]
        if c["mode"] == "pixelwise":
            _call("mlf_summary_image_device", state["movie"], c["h"], c["w"], c["t"], c["w1"], c["w2"], 3, 5,
                  o["image"], o["spatial"], o["temporal"])
        else:
            _call("mlf_summary_image_global_device", state["movie"], c["h"], c["w"], c["t"], 5, o["image"],
                  o["spatial"], o["temporal"])
    else:
        _call("mlf_rectify_device", state["frames"], c["h"], c["w"], c["t"], 8.3, 7.9, N, c["dx"], state["out"])
    return state["out"]


# ------------------------------------------------- what a pass cannot do without
def _taps(planes):
    """Kernel pixels of one view over all planes."""
    return sum((30 * _radius(z) + 1) ** 2 for z in _z_um(planes))


def work(case):
    kind = case["kind"]
    if kind in ("rl", "recon", "batch"):
        grids = _grids(case) if kind == "batch" else [(case["n1"], case["n2"])]
        steps = 177 * case["iters"]
        cells = sum(a * b for a, b in grids)
        volume = 4.0 * cells * NP * case["planes"]
        taps = 177 * _taps(case["planes"])
        wide = 4 if case["prec"] == "fp32" else 2
        # every view step needs the volume that the one before it wrote: a
        # volume beyond the caches is read and written once per step
        passes = 2 * steps if volume > VOLUME_CACHE else 1
        out = 8 if kind == "recon" else 4
        return {"flops": 4.0 * steps * cells * _taps(case["planes"]),
                "bytes": volume * passes + 2.0 * wide * taps + 4.0 * cells * NP + volume / 4 * out}
    if kind == "project":
        cells = case["n1"] * case["n2"]
        wide = 4 if case["prec"] == "fp32" else 2
        return {"flops": 2.0 * 177 * cells * _taps(case["planes"]),
                "bytes": 4.0 * cells * NP * (case["planes"] + 1) + wide * 177.0 * _taps(case["planes"])}
    if kind == "mex":
        px = case["w"] * case["h"] * case["n"]
        return {"flops": 2.0 * px * case["kw"] ** 2, "bytes": 8.0 * px + 4.0 * NP * case["kw"] ** 2}
    if kind == "seedlib":
        n = case["segments"] * (0.25 * case["z"] + 0.75)  # slices, on average
        px = case["w"] * case["h"]
        return {"flops": 2.0 * px * n * case["kw"] ** 2,
                "bytes": 4.0 * px * (n + case["segments"]) + 4.0 * NP * case["z"] * case["kw"] ** 2}
    if kind == "summary":
        px, t = case["h"] * case["w"], case["t"]
        # the rank-1 background is 5 dependent rounds over the movie
        reads = 6 if 4 * px * t > VOLUME_CACHE else 1
        return {"flops": 30.0 * px * t, "bytes": 4.0 * px * t * reads + 16.0 * px}
    px = case["h"] * case["w"] * case["t"]
    return {"flops": 10.0 * px, "bytes": 8.0 * px}


# -------------------------------------------------- the results in 64 bits
class _Exact:
    """Forward and backward projection, update and low-pass filter of one patch
    in 64 bits, planes of one radius together: volume [n1 n2, planes, 225] per
    radius, taps [k1 k2, planes, 225]."""

    def __init__(self, n1, n2, planes, device):
        self.n1, self.n2, self.planes, self.dev = n1, n2, planes, device
        z_um = _z_um(planes)
        self.radii = sorted({_radius(z) for z in z_um})
        self.of = {r: [i for i, z in enumerate(z_um) if _radius(z) == r] for r in self.radii}
        self.block = [(2 * _radius(z) + 1) ** 2 * NP for z in z_um]
        self.tabs = torch.from_numpy(_tables(planes)).to(device)
        self.scale = 1.0

    def taps(self, k):
        o = k * sum(self.block)
        z_um, out = _z_um(self.planes), {r: [] for r in self.radii}
        for zi, n in enumerate(self.block):
            r = _radius(z_um[zi])
            K = 2 * r + 1
            out[r].append(self.tabs[o:o + n].reshape(K, K, NP).transpose(0, 1).reshape(K * K, NP))
            o += n
        return {r: torch.stack(t, 1).double().reshape(-1, len(t) * NP) * self.scale for r, t in out.items()}

    def split(self, vol):  # [I1, I2, planes] -> per radius [n1 n2, planes * 225]
        v = vol.reshape(self.n1, N, self.n2, N, self.planes).permute(0, 2, 4, 3, 1)
        return {r: v[:, :, self.of[r]].reshape(self.n1 * self.n2, -1).contiguous() for r in self.radii}

    def join(self, X):
        v = torch.empty((self.n1, self.n2, self.planes, N, N), device=self.dev, dtype=torch.float64)
        for r in self.radii:
            v[:, :, self.of[r]] = X[r].reshape(self.n1, self.n2, -1, N, N)
        return v.permute(0, 4, 1, 3, 2).reshape(N * self.n1, N * self.n2, self.planes)

    def forward(self, X, W):
        y = torch.zeros((self.n1, self.n2), device=self.dev, dtype=torch.float64)
        for r in self.radii:
            K = 2 * r + 1
            q = W[r] @ X[r].T  # [k1 k2, n1 n2]
            full = torch.nn.functional.fold(q[None], (self.n1 + 2 * r, self.n2 + 2 * r), K)
            y += full[0, 0, r:r + self.n1, r:r + self.n2]
        return y

    def backward(self, R, W, r):
        cols = torch.nn.functional.unfold(R[None, None], 2 * r + 1, padding=r)[0]  # [k1 k2, n1 n2]
        return cols.T @ W[r]

    def filter(self, vol):
        planes = self.planes
        nf = 3 * (math.ceil(planes / 3) + math.ceil(planes / 3) % 2)
        half = math.floor(planes / 2 + 0.5)
        axis = np.arange(1, nf + 1) - nf / 2.0
        omega = np.maximum(8 * np.exp(-(axis / 100.0 * 2 * math.sqrt(math.log(2))) ** 2), 0.2)

        def bank(size, w):
            g = np.abs(np.fft.fft(np.exp(-(((np.arange(1, size + 1) - size / 2.0) / w) ** 2))))
            return torch.from_numpy(g / g.max()).to(self.dev)

        for z in range(planes):
            if not half - nf / 2.0 + 1 <= z + 1 <= half + nf / 2.0:
                continue
            w = omega[int(z + 1 - half + nf / 2.0) - 1]
            img = vol[:, :, z]
            f = torch.fft.fft2(img) * bank(vol.shape[0], w)[:, None] * bank(vol.shape[1], w)[None, :]
            out = torch.fft.ifft2(f).real
            vol[:, :, z] = img.sum() * out / out.sum()
        return vol

    def reconstruct(self, image, weights, iters):
        im = torch.from_numpy(image).to(self.dev).double()
        vol = torch.full((N * self.n1, N * self.n2, self.planes), 1.0, device=self.dev, dtype=torch.float64)
        X = self.split(vol / vol.numel() * im.sum())
        ones = torch.ones((self.n1, self.n2), device=self.dev, dtype=torch.float64)
        for _ in range(iters):
            for k, (u, v) in enumerate(_views()):
                W, w = self.taps(k), weights[k]
                R = im[u::N, v::N] / self.forward(X, W)
                R = torch.where(torch.isfinite(R), R, torch.zeros_like(R))
                for r in self.radii:
                    c = X[r] * self.backward(R, W, r) / self.backward(ones, W, r)
                    c = torch.where(torch.isfinite(c) & (c >= 0), c, torch.zeros_like(c))
                    X[r] = (c * w + (1 - w) * X[r]).clamp_(min=0)
            X = self.split(self.filter(self.join(X)))
        return self.join(X)


def _exact_mex(x, k):
    """[n, h, w] correlation with [15, 15, kw, kw] kernels by output phase."""
    n, h, w = x.shape
    kw = k.shape[-1]
    size = (h + kw - 1, w + kw - 1)
    out = torch.empty(x.shape, device=x.device, dtype=torch.float64)
    for i in range(0, n, 16):
        fx = torch.fft.rfft2(x[i:i + 16].double(), s=size)
        for q in range(min(N, h)):
            fk = torch.fft.rfft2(k[q].double(), s=size).conj()
            for p in range(min(N, w)):
                full = torch.fft.irfft2(fx * fk[p], s=size).roll((kw // 2, kw // 2), (1, 2))
                out[i:i + 16, q::N, p::N] = full[:, q:h:N, p:w:N]
    return out


def _movmean(x, k):
    a, b = ((k - 1) // 2, (k - 1) // 2) if k % 2 else (k // 2, k // 2 - 1)
    t = x.shape[0]
    sums = torch.cat([torch.zeros_like(x[:1]), x.cumsum(0)])
    j = torch.arange(t, device=x.device)
    lo, hi = (j - a).clamp(min=0), (j + b).clamp(max=t - 1)
    return (sums[hi + 1] - sums[lo]) / (hi - lo + 1).double()[:, None]


def _exact_summary(case, movie):
    t = case["t"]
    y = movie.reshape(t, -1)
    mx = y.max().double()
    # 'global' divides the movie first, 'pixelwise' the products: the same in exact arithmetic
    s = torch.full((y.shape[1],), 1.0 / math.sqrt(y.shape[1]), device=y.device, dtype=torch.float64)
    for it in range(5):
        b = torch.stack([(f.double() * s).sum() for f in y]) / mx
        b = b / b.norm()
        s = torch.zeros_like(s)
        for j in range(t):
            s += y[j].double() * b[j]
        s /= mx
        if it < 4:
            s = s / s.norm()
    img = torch.empty_like(s)
    for i in range(0, y.shape[1], 65536):
        x = y[:, i:i + 65536].double() / mx
        if case["mode"] == "pixelwise":
            v = _movmean(x - _movmean(x, case["w1"]), case["w2"]) ** 3
            img[i:i + 65536] = torch.sqrt((v * v).sum(0) / t - v.mean(0) ** 2)
        else:
            a, m, y1, c = (x * x).sum(0), x.mean(0), s[i:i + 65536], b.mean()
            img[i:i + 65536] = torch.sqrt((a - y1 ** 2) / t - m ** 2 + 2 * m * y1 * c - y1 ** 2 * c ** 2)
    good = img[~torch.isnan(img)]
    shape = (case["w"], case["h"])
    return {"image": (img / good.max()).reshape(shape), "spatial": s.reshape(shape), "temporal": b}


def _exact_rectify(case, frames):
    def axis(centre, size):
        step = case["dx"] / N
        down = centre - step * np.arange(int(math.floor((centre + step) / step + 1e-10)) + 1)
        up = centre + step + step * np.arange(int(math.floor((size + 0.9 - centre - step) / step + 1e-10)) + 1)
        grid = np.concatenate([down[::-1], up])
        first = len(down) - N // 2
        q = grid[first - N * (first // N):]
        return torch.from_numpy(q[:N * (len(q) // N)]).to(frames.device)

    xq, yq = axis(8.3, case["w"]), axis(7.9, case["h"])
    kx, ky = xq.floor().long().clamp(1, case["w"] - 1), yq.floor().long().clamp(1, case["h"] - 1)
    tx, ty = (xq - kx)[:, None], (yq - ky)[None, :]
    out = torch.empty((case["t"], len(xq), len(yq)), device=frames.device, dtype=torch.float64)
    for j in range(case["t"]):
        f = frames[j].double()
        a, b = f[kx - 1], f[kx]
        out[j] = (1 - tx) * ((1 - ty) * a[:, ky - 1] + ty * a[:, ky]) + tx * ((1 - ty) * b[:, ky - 1] + ty * b[:, ky])
    return out


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if work(case)["flops"] > 2e14 and kind in ("rl", "batch"):
        return None  # over 20 s in 64 bits
    if kind in ("rl", "batch"):
        grids = _grids(case) if kind == "batch" else [(case["n1"], case["n2"])]
        images = [_image(rng, a, b, case["planes"]) for a, b in grids]
        vols = [_Exact(a, b, case["planes"], "cuda").reconstruct(im, [0.3] * 177, case["iters"]).cpu().numpy()
                for (a, b), im in zip(grids, images)]
        return vols if kind == "batch" else vols[0]
    if kind == "recon":
        e = _Exact(case["n1"], case["n2"], case["planes"], "cuda")
        # every depth of H sums to one; a view's weight follows its share of the sum
        H, _ = _dense(case["planes"])
        depth = [float(H[:, :, :, :, z].sum(dtype=np.float64)) for z in range(case["planes"])]
        z_um = _z_um(case["planes"])
        o, share, tabs = 0, np.zeros((N, N)), e.tabs.double()
        for u, v in _views():
            for zi, n in enumerate(e.block):
                tabs[o:o + n] /= depth[zi]
                share[u, v] += float(tabs[o:o + n].sum())
                o += n
        e.tabs = tabs
        share = share / share.sum()
        share = (share - share.min()) / (share - share.min()).max()
        weights = [0.3 * share[u, v] for u, v in _views()]
        assert len(z_um) == len(depth)
        return e.reconstruct(_image(rng, case["n1"], case["n2"], case["planes"]), weights, case["iters"]).cpu().numpy()
    if kind == "project":
        e = _Exact(case["n1"], case["n2"], case["planes"], "cuda")
        vol = torch.from_numpy(_volume(rng, case["n1"], case["n2"], case["planes"])).to("cuda").double()
        X = e.split(vol)
        out = torch.zeros((N * case["n1"], N * case["n2"]), device="cuda", dtype=torch.float64)
        for k, (u, v) in enumerate(_views()):
            out[u::N, v::N] = e.forward(X, e.taps(k))
        return out.cpu().numpy()
    if kind == "mex":
        g = _gen(seed)
        x = _bitmaps(g, case["w"], case["h"], case["n"])
        return _exact_mex(x, _mex_kernels(g, case["kw"], 1)[0])
    if kind == "seedlib":
        g = _gen(seed)
        planes, ptr = _segments(case, seed)
        x = _bitmaps(g, case["w"], case["h"], len(planes))
        k = _mex_kernels(g, case["kw"], case["z"])
        out = torch.zeros((case["segments"], case["h"], case["w"]), device="cuda", dtype=torch.float64)
        for z in range(case["z"]):
            at = [i for i, p in enumerate(planes) if p == z]
            if at:
                seg = [next(s for s in range(case["segments"]) if ptr[s] <= i < ptr[s + 1]) for i in at]
                out.index_add_(0, torch.tensor(seg, device="cuda"), _exact_mex(x[at], k[z]))
        return out
    if kind == "summary":
        return _exact_summary(case, _movie(_gen(seed), case["h"], case["w"], case["t"]))
    return _exact_rectify(case, _movie(_gen(seed), case["h"], case["w"], case["t"]))
