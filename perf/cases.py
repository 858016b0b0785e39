"""Performance cases of the drift-correction library.

Each case is work that a user of the library has it do, through the ctypes
binding of the C ABI (motioncorr1exp_amd): whole movies from frames resident
in device memory (mc_align_movie, mc_align_batch), the stage entry points on
resident spectra (mc_pair_shifts, mc_sharpness) and the transforms of the
cufunc.h seam (mc_fft2d, mc_ifft2d).  exact() restates the same algorithm in
FP64 with torch and numpy only.

Movies are seeded random-field phantoms (power 1/(1 + (k/0.05)^2)) under a
random-walk drift with Poisson counts, as the tests and the benchmark use.
The drift moves in whole steps of the peak search's grid (1/32 transform
pixel), so that the picked grid point is not decided by the last bits of a
near tie and the picked shifts can be compared exactly.  For the same reason
small frames carry a higher dose (coarser fractions).
"""
import ctypes
import math
import os

import numpy as np
import torch

import motioncorr1exp_amd as mc

TUNE_TABLE = os.path.join(os.path.dirname(os.path.abspath(mc.__file__)), "tune_mi355x.jsonl")

MOVIE = dict(kind="movie", nx=0, ny=0, frames=0, dtype="uint8", dose=1.0, pad=0, bin=1.0, fod=2,
             bft=150.0, box=96, itr=0, precision=0, gain=False, tuned=False)


def _movie(name, **kw):
    return dict(MOVIE, name=name, **kw)


def listed():
    return [
        # One small movie at a time, where launches, copies and host work count:
        # a 512 x 512 x 10 float stack, every pair, no iteration.
        _movie("small-512x10", nx=512, ny=512, frames=10, dtype="float32", dose=12.0, fod=4),
        # The headline workload: a K2 counting movie as float, padded to 4096,
        # by a service that loads the shipped launch table at start-up.
        _movie("k2-pad4096x40", nx=3838, ny=3710, frames=40, dtype="float32", dose=0.8, pad=4096,
               tuned=True),
        # The same detector as the command line runs it by default: raw bytes and
        # a gain reference, the square crop (n = 3710), with -itr 3.
        _movie("k2-crop3710x24", nx=3838, ny=3710, frames=24, gain=True, itr=3),
        # 8-bit counts binned 2x, all 276 pairs, three align-to-sum rounds, with
        # the library's default launch shapes.
        _movie("bin2-4096x24", nx=4096, ny=4096, frames=24, bin=2.0, fod=11, itr=3),
        # A K3 movie at its default square crop (n = 4092), 16-bit.
        _movie("k3-crop4092x16", nx=5760, ny=4092, frames=16, dtype="int16"),
        # A transform size with no radix plan (1854 = 2 9 103), 16-bit, one round.
        _movie("crop1854x20", nx=1900, ny=1854, frames=20, dtype="uint16", itr=1),
        # Super-resolution K2 frames binned 2x (canvas 7420, n = 3710): the
        # largest frames that one movie brings.
        _movie("k2-super-bin2x12", nx=7676, ny=7420, frames=12, dose=0.5, bin=2.0),
        # The precision form (hi/lo matrix products in the pair stage).
        _movie("hilo-2048x20", nx=2000, ny=1960, frames=20, pad=2048, precision=1),
        # A service aligning movies of uneven size and length in one call.
        dict(name="batch-8", kind="batch", movies=8, side_lo=1024, side_hi=4096, frames_lo=8,
             frames_hi=50, pick=7, itr=3, tuned=True),
        # Pair shifts and box maps on resident spectra, a smaller peak box.
        dict(name="pairs-1536-box64", kind="pairs", n=1536, frames=20, box=64, bft=150.0, fod=2,
             dose=2.0),
        # Sharpness of the aligned sum and its adjoint gradient (one step of a
        # gradient refinement driven by the caller).
        dict(name="sharpness-2048x24", kind="sharpness", n=2048, frames=24, bft=150.0, dose=1.0),
        # The 2-D transforms of the cufunc.h seam, both directions.
        dict(name="fft-1000", kind="fft", n=1000),
    ]


def _log_int(rng, lo, hi, even=False):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return v // 2 * 2 if even else v


def _dose(rng, side):
    """0.5 to 1.5 counts per pixel and frame, more on frames below 1500."""
    return round(max(rng.uniform(0.5, 1.5), min(12.0, 1.5 * (1500 / side) ** 2)), 2)


# canvases of the pad geometry (sizes with a radix plan)
PADS = (512, 768, 1024, 1280, 1536, 1920, 2048, 2560, 3072, 3840, 4096)


def draw(rng):
    kind = rng.choice(["pad", "pad", "crop", "crop", "bin", "hilo", "batch", "pairs", "sharpness",
                       "fft"])
    dtype = rng.choice(["uint8", "int8", "int16", "uint16", "float32"])
    box = rng.choice([64, 96, 96, 96, 128])
    itr = rng.choice([0, 0, 1, 3])
    if kind == "pad":
        pad = rng.choice(PADS)
        nx = rng.randint(pad * 7 // 8, pad)
        ny = rng.randint(pad * 7 // 8, pad)
        return dict(MOVIE, nx=nx, ny=ny, frames=_log_int(rng, 8, 40), dtype=dtype,
                    dose=_dose(rng, min(nx, ny)), pad=pad, box=box, fod=rng.randint(1, 4), itr=itr,
                    tuned=rng.random() < 0.5)
    if kind == "crop":  # the default square crop of any frame
        big = rng.random() < 0.3
        nx = _log_int(rng, 400, 2600) if not big else 3838
        ny = max(400, nx - rng.randint(0, nx // 8)) if not big else 3710
        return dict(MOVIE, nx=nx, ny=ny, frames=_log_int(rng, 8, 32), dtype=dtype,
                    dose=_dose(rng, ny), box=box, fod=rng.randint(1, 4), itr=itr,
                    gain=rng.random() < 0.5)
    if kind == "bin":
        nx = _log_int(rng, 1000, 4200)
        ny = max(1000, nx - rng.randint(0, nx // 8))
        return dict(MOVIE, nx=nx, ny=ny, frames=_log_int(rng, 8, 24), dtype=dtype,
                    dose=_dose(rng, ny), bin=rng.choice([1.5, 2.0, 2.0]), fod=rng.randint(1, 8),
                    itr=itr)
    if kind == "hilo":
        pad = rng.choice([512, 1024, 1536, 2048, 2560, 3072, 4096])
        nx, ny = rng.randint(pad * 7 // 8, pad), rng.randint(pad * 7 // 8, pad)
        return dict(MOVIE, nx=nx, ny=ny, frames=_log_int(rng, 8, 24), dtype=dtype,
                    dose=_dose(rng, min(nx, ny)), pad=pad, precision=1)
    if kind == "batch":
        return dict(kind="batch", movies=rng.randint(2, 8), side_lo=1024, side_hi=4096, frames_lo=8,
                    frames_hi=30, pick=rng.randint(0, 1 << 20), itr=rng.choice([0, 1, 3]),
                    tuned=rng.random() < 0.5)
    if kind == "pairs":
        n = _log_int(rng, 400, 4200, even=True)
        return dict(kind="pairs", n=n, frames=rng.randint(6, 24), box=rng.choice([32, 64, 96, 128]),
                    bft=rng.choice([100.0, 150.0, 500.0]), fod=rng.randint(1, 3),
                    dose=_dose(rng, n))
    if kind == "sharpness":
        return dict(kind="sharpness", n=_log_int(rng, 256, 4096, even=True),
                    frames=rng.randint(6, 32), bft=150.0, dose=1.0)
    return dict(kind="fft", n=_log_int(rng, 64, 8192, even=True))


# ------------------------------------------------------------------ inputs
class _Dev:
    """A torch tensor as the binding's device arrays: an object with .ptr."""

    def __init__(self, t):
        self.tensor = t
        self.ptr = t.data_ptr()


def _smooth5(m):
    while True:
        k = m
        for f in (2, 3, 5):
            while k % f == 0:
                k //= f
        if k == 1 and m % 2 == 0:
            return m
        m += 1


def _drift(frames, seed, bin_=1.0, step=0.7):
    """Random-walk positions (frame pixels) on the 1/32 grid of the binned image."""
    steps = np.random.default_rng(seed + 7919).normal(0.0, step, size=(frames, 2))
    steps[0] = 0.0
    return np.round(np.cumsum(steps, axis=0) / bin_ * 32) / 32 * bin_


def _phantom(m, dose, gen):
    """Spectrum of an m x m random-field phantom with mean `dose`."""
    f = torch.fft.rfft2(torch.randn(m, m, generator=gen, device="cuda"))
    ky = torch.fft.fftfreq(m, device="cuda")[:, None]
    kx = torch.fft.rfftfreq(m, device="cuda")[None, :]
    f = f * (1.0 / (1.0 + (kx * kx + ky * ky) / 0.05 ** 2)).sqrt()
    f[0, 0] = 0
    g = torch.fft.irfft2(f, s=(m, m))
    g = (g - g.mean()) / g.std()
    return torch.fft.rfft2(torch.exp(0.8 * g - 0.32) * dose), kx, ky


def _frames(nx, ny, frames, dtype, dose, seed, bin_=1.0):
    """frames x ny x nx counts of `dtype` on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    m = _smooth5(max(nx, ny) + 64)
    P, kx, ky = _phantom(m, dose, gen)
    t = _drift(frames, seed, bin_)
    out = torch.empty(frames, ny, nx, dtype=getattr(torch, dtype), device="cuda")
    for f in range(frames):
        ph = torch.exp(-2j * math.pi * ky * t[f, 1]) * torch.exp(-2j * math.pi * kx * t[f, 0])
        img = torch.fft.irfft2(P * ph, s=(m, m))[:ny, :nx].clamp_(min=0).contiguous()
        counts = torch.poisson(img, generator=gen)
        if dtype != "float32":  # counts saturate
            counts.clamp_(max=torch.iinfo(out.dtype).max)
        out[f] = counts.to(out.dtype)
    return out


def _gain(nx, ny, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed + 31)
    return 1.0 + 0.05 * torch.randn(ny, nx, generator=gen, device="cuda")


def _spectra(n, frames, seed, dose):
    """frames x n x (n/2+1) complex64 spectra of a movie (host)."""
    x = _frames(n, n, frames, "float32", dose, seed)
    out = np.empty((frames, n, n + 2), np.float32)
    for f in range(frames):
        s = torch.fft.rfft2(x[f].double()).to(torch.complex64)
        out[f] = torch.view_as_real(s).reshape(n, n + 2).cpu().numpy()
    return out


def _batch_movies(case):
    """The uneven movies of a batch case: sides, frames and doses from `pick`,
    each padded to the next canvas."""
    rng = np.random.default_rng(case["pick"])
    out = []
    for i in range(case["movies"]):
        side = int(rng.integers(case["side_lo"], case["side_hi"] + 1))
        F = int(rng.integers(case["frames_lo"], case["frames_hi"] + 1))
        pad = next(p for p in PADS if p >= side)
        dose = max(float(rng.uniform(0.5, 1.5)), 1.5 * (1500 / side) ** 2)
        out.append(dict(MOVIE, nx=side, ny=side, frames=F, dose=dose, pad=pad, itr=case["itr"]))
    return out


_contexts = {}


def _context(tuned):
    """The context that a program keeps for all its movies."""
    if tuned not in _contexts:
        _contexts[tuned] = mc.Context(0)
        if tuned:
            _contexts[tuned].tune_load(TUNE_TABLE)
    return _contexts[tuned]


def _size(case):
    """(unbinned canvas, transform size) of a movie case."""
    if case["pad"]:
        nu = case["pad"]
    else:
        nu = min(case["nx"], case["ny"])
        nu = nu // 4 * 4 if case["bin"] == 2.0 else nu // 2 * 2
    return nu, int(np.float32(nu) / np.float32(case["bin"])) // 2 * 2


def _prepare_movie(case, seed):
    F = case["frames"]
    n = _size(case)[1]
    st = dict(frames=_Dev(_frames(case["nx"], case["ny"], F, case["dtype"], case["dose"], seed,
                             case["bin"])),
              shape=(F, case["ny"], case["nx"]), dtype=np.dtype(case["dtype"]),
              sum=_Dev(torch.empty(n, n, device="cuda")), corr=None,
              params=mc.default_params(F, pad=case["pad"], bin=case["bin"],
                                       FrameDistOffset=case["fod"], bfactor=case["bft"],
                                       CCPeakSearchDim=case["box"], iter=case["itr"],
                                       precision=case["precision"]))
    if case["gain"]:
        st["gain"] = _Dev(_gain(case["nx"], case["ny"], seed))
        st["corr"] = mc.corrections(gain=st["gain"])
    return st


WANT = ("pair_b", "final_shift", "frame_shift")


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind)
    if kind == "movie":
        st.update(_prepare_movie(case, seed), ctx=_context(case["tuned"]))
    elif kind == "batch":
        movies = [_prepare_movie(m, seed * 64 + i) for i, m in enumerate(_batch_movies(case))]
        st.update(ctx=_context(case["tuned"]), movies=movies,
                  items=[dict(dev=m["frames"], shape=m["shape"], dtype=m["dtype"],
                              params=m["params"], want=WANT, sum_dev=m["sum"]) for m in movies])
    elif kind in ("pairs", "sharpness"):
        F, n = case["frames"], case["n"]
        st["ctx"] = mc.Context(0)  # its spectra stay resident from pass to pass
        st["ctx"].set_spectra(_spectra(n, F, seed, case["dose"]))
        st["bft"] = case["bft"]
        if kind == "pairs":
            st["pairs"], st["box"] = mc.pair_list(F, case["fod"]), case["box"]
        else:
            t = _drift(F, seed)
            st["shift"] = -t + np.random.default_rng(seed).normal(0.0, 0.1, t.shape)
    else:
        n = case["n"]
        gen = torch.Generator(device="cuda").manual_seed(seed)
        st["image"] = torch.zeros(n, n + 2, device="cuda")
        st["image"][:, :n] = torch.poisson(torch.ones(n, n, device="cuda"), generator=gen)
        other = torch.poisson(torch.ones(n, n, device="cuda"), generator=gen)
        spec = torch.fft.rfft2(other.double()).to(torch.complex64)
        st["spec"] = torch.view_as_real(spec).reshape(n, n + 2).contiguous()
        st["fwd"], st["inv"] = torch.empty_like(st["image"]), torch.empty_like(st["image"])
        st["n"], st["plans"] = n, _Plans(n)
    torch.cuda.synchronize()
    return st


class _Plans:
    """The forward and inverse plan of one size (GPUFFTPlan, GPUIFFTPlan)."""

    def __init__(self, n):
        self.L = mc.lib()
        self.fwd, self.inv = ctypes.c_void_p(), ctypes.c_void_p()
        mc.check(self.L.mc_fft_plan(ctypes.byref(self.fwd), n))
        mc.check(self.L.mc_ifft_plan(ctypes.byref(self.inv), n))

    def __del__(self):
        self.L.mc_fft_destroy(self.fwd)
        self.L.mc_fft_destroy(self.inv)


def run(st):
    kind = st["kind"]
    if kind == "movie":
        r = st["ctx"].align_movie(st["frames"], st["shape"], st["dtype"], st["params"], want=WANT,
                                  sum_dev=st["sum"], corr=st["corr"])
        return {k: r[k] for k in WANT} | {"sum": st["sum"].tensor}
    if kind == "batch":
        res, _ = st["ctx"].align_batch(st["items"])
        return [{k: r[k] for k in WANT} | {"sum": m["sum"].tensor}
                for r, m in zip(res, st["movies"])]
    if kind == "pairs":
        b, cc, boxes = st["ctx"].pair_shifts(st["pairs"], st["bft"], st["box"], want_boxes=True)
        # cc is a value of the float32 box map, carried in a double
        return {"b": b, "cc": cc.astype(np.float32), "boxes": boxes}
    if kind == "sharpness":
        J, g = st["ctx"].sharpness(st["shift"], st["bft"])
        return {"J": J, "grad": g}
    L, p, nb = st["plans"].L, st["plans"], st["image"].numel() * 4
    # in-place transforms: the caller's data is copied in first
    mc.check(L.mc_mem_d2d(st["fwd"].data_ptr(), st["image"].data_ptr(), nb))
    mc.check(L.mc_fft2d(st["fwd"].data_ptr(), p.fwd))
    mc.check(L.mc_mem_d2d(st["inv"].data_ptr(), st["spec"].data_ptr(), nb))
    mc.check(L.mc_ifft2d(st["inv"].data_ptr(), p.inv))
    return {"spectrum": st["fwd"], "image": st["inv"][:, :st["n"]]}


# ------------------------------------------------------------------- work
def _pairs_of(F, fod):
    d = F // 2 - fod
    d = 1 if d <= 0 else min(d, F // 2)
    return [(i, j) for i in range(F) for j in range(i + d, F)]


def _pair_flops(P, n, box):
    """Per (pair, column): product and weight, and an inverse of n points of
    which box are kept (n log2(128) plus the box rows from n/128 terms); then
    the row product to box x box."""
    H = n // 2 + 1
    return P * H * (9 * n + 5 * n * 7 + box * (n / 128) * 8 + 4 * box * box)


def _movie_work(case):
    """The spectra of a movie (several GB) do not fit on the chip: they are
    written once and read once by each stage that needs all of them (pairs,
    two passes per round, final sum)."""
    F, es = case["frames"], np.dtype(case["dtype"]).itemsize
    nu, n = _size(case)
    w, h = (min(case["nx"], nu), min(case["ny"], nu)) if case["pad"] else (nu, nu)
    S = 8 * n * (n // 2 + 1)
    P = len(_pairs_of(F, case["fod"]))
    itr = case["itr"]
    by = F * w * h * es + F * S * (3 + 2 * itr) + 4 * n * n
    fl = F * (h * 2.5 * nu * math.log2(nu) + (n // 2 + 1) * 5 * nu * math.log2(nu))
    fl += _pair_flops(P + itr * F, n, case["box"])
    fl += (1 + itr) * F * (n // 2 + 1) * n * 8 + 2.5 * n * n * math.log2(n) * 2
    return {"bytes": by, "flops": fl}


def work(case):
    kind = case["kind"]
    if kind == "movie":
        return _movie_work(case)
    if kind == "batch":
        ws = [_movie_work(m) for m in _batch_movies(case)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    n = case["n"]
    S = 8 * n * (n // 2 + 1)
    if kind == "pairs":
        P = len(_pairs_of(case["frames"], case["fod"]))
        return {"bytes": case["frames"] * S + 4 * P * case["box"] ** 2,
                "flops": _pair_flops(P, n, case["box"])}
    if kind == "sharpness":  # the sum, then the gradient against it
        F = case["frames"]
        return {"bytes": 2 * F * S, "flops": 2 * F * (S / 8) * 16}
    return {"bytes": 4 * S, "flops": 2 * 5 * n * n * math.log2(n)}


# ---------------------------------------------- the same in 64 bits (torch)
C128 = torch.complex128


def _x_index(n):
    """(kx, y') of a half spectrum of size n: y' = ky or ky - n."""
    kx = torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64)
    y = torch.arange(n, device="cuda", dtype=torch.float64)
    return kx, torch.where(y < n // 2, y, y - n)


def _crop_bins(s, nu, n):
    """Fourier crop of an nu half spectrum to n."""
    if n == nu:
        return s
    return torch.cat([s[: n // 2, : n // 2 + 1], s[nu - n // 2:, : n // 2 + 1]])


def _exact_spectra(case, x, gain=None):
    nu, n = _size(case)
    out = []
    for f in range(case["frames"]):
        v = x[f].float()
        if gain is not None:
            v = v * gain  # the reference corrects frames in float
        if case["pad"]:
            v = v[:nu, :nu].double()
            c = torch.full((nu, nu), float(v.mean()), dtype=torch.float64, device="cuda")
            c[: v.shape[0], : v.shape[1]] = v
        else:
            c = v[:nu, :nu].double()
        out.append(_crop_bins(torch.fft.rfft2(c), nu, n).clone())
    return out


class _Box:
    """Central box of the weighted correlation maps of size n."""

    def __init__(self, n, box, bft):
        self.n, self.ori, self.box = n, (n - box) // 2, box
        kx, y = _x_index(n)
        m = -0.5 * bft / n / n
        sgn = 1.0 - 2.0 * ((kx[None, :] + y[:, None]) % 2)
        self.z = sgn * torch.exp(m * (kx[None, :] ** 2 + y[:, None] ** 2)) / (n * (n // 2 + 1))
        c = torch.arange(self.ori, self.ori + box, device="cuda")
        k = torch.arange(n // 2 + 1, device="cuda")
        t = 2 * math.pi * ((k[:, None] * c[None, :]) % n).double() / n
        a = torch.full((n // 2 + 1, 1), 2.0, dtype=torch.float64, device="cuda")
        a[0] = a[-1] = 1.0
        self.cos, self.sin = a * torch.cos(t), a * torch.sin(t)

    def __call__(self, a, b):
        t = torch.fft.ifft(a * b.conj() * self.z, dim=0, norm="forward")
        t = t[self.ori: self.ori + self.box]
        return t.real @ self.cos - t.imag @ self.sin


def _exact_peak(m, n):
    """FindShift of the reference on one box map (cufunc.cu:396-497)."""
    B = m.shape[0]
    i = int(torch.argmax(m.reshape(-1)))
    o = [min(max(v - 8, 0), B - 16) for v in (i % B, i // B)]
    g = torch.fft.rfft2(m[o[1]: o[1] + 16, o[0]: o[0] + 16])
    kx = torch.arange(9, device="cuda", dtype=torch.float64)
    ky = torch.fft.fftfreq(16, 1 / 16, device="cuda", dtype=torch.float64)
    r = torch.floor(torch.sqrt(kx[None, :] ** 2 + ky[:, None] ** 2))
    g = g * torch.where(r < 8, torch.cos(math.pi * r / 8) / 2 + 0.5, torch.zeros_like(r))
    p = torch.arange(512, device="cuda", dtype=torch.float64)
    g = torch.exp(2j * math.pi * ((p[:, None] * ky) % 512) / 512) @ g
    a = torch.full((9, 1), 2.0, dtype=torch.float64, device="cuda")
    a[0] = 1.0
    t = 2 * math.pi * ((kx[:, None] * p) % 512) / 512
    u = g.real @ (a * torch.cos(t)) - g.imag @ (a * torch.sin(t))
    i = int(torch.argmax(u.reshape(-1)))
    return (o[0] + (i % 512) / 32 - B // 2, o[1] + (i // 512) / 32 - B // 2,
            float(u.reshape(-1)[i]) / n / n / 256)


def _solve(pairs, F, b):
    A = np.zeros((len(pairs), F - 1))
    for q, (i, j) in enumerate(pairs):
        A[q, i:j] = 1
    return A, np.linalg.lstsq(A, b, rcond=None)[0]


def _connected(pairs, F):
    group = list(range(F))

    def root(v):
        while group[v] != v:
            v = group[v]
        return v

    for i, j in pairs:
        group[root(i)] = root(j)
    return len({root(v) for v in range(F)}) == 1


def _exact_drift(pairs, F, b, kit=1.0):
    """Least squares, outlier rejection, least squares (mfunc.h:50-146)."""
    A, s = _solve(pairs, F, b)
    ki = np.hypot(*(A @ s - b).T)
    order = np.argsort(ki, kind="stable")
    i = len(pairs) - 1
    while i >= F - 1 and ki[order[i]] >= kit:
        i -= 1
    while True:
        good = np.sort(order[: i + 1])
        i += 1
        if _connected([pairs[g] for g in good], F) or i >= len(pairs):
            break
    return _solve([pairs[g] for g in good], F, b[good])[1]


def _exact_sum(specs, n, shifts):
    kx, y = _x_index(n)
    acc = torch.zeros(n, n // 2 + 1, dtype=C128, device="cuda")
    for s, (sx, sy) in zip(specs, shifts):
        acc += s * (torch.exp(2j * math.pi * ((sy * y[:, None] / n) % 1.0))
                    * torch.exp(2j * math.pi * ((sx * kx[None, :] / n) % 1.0)))
    return acc


def _exact_image(spec, n):
    """C2R with the DC and Nyquist columns' imaginary parts ignored, / n^2."""
    t = torch.fft.ifft(spec, dim=0)
    t[:, 0].imag.zero_()
    t[:, -1].imag.zero_()
    return torch.fft.irfft(t, n=n, dim=1)


def _exact_movie(case, seed):
    F, n = case["frames"], _size(case)[1]
    x = _frames(case["nx"], case["ny"], F, case["dtype"], case["dose"], seed, case["bin"])
    specs = _exact_spectra(case, x, _gain(case["nx"], case["ny"], seed) if case["gain"] else None)
    del x
    box = _Box(n, case["box"], case["bft"])
    pairs = _pairs_of(F, case["fod"])
    b = np.array([_exact_peak(box(specs[i], specs[j]), n)[:2] for i, j in pairs])
    s = _exact_drift(pairs, F, b)
    pos = np.vstack([np.zeros((1, 2)), np.cumsum(s, axis=0)])
    for _ in range(case["itr"]):
        total = _exact_sum(specs, n, -pos)
        new = np.array([_exact_peak(box(total, f), n)[:2] for f in specs])
        pos = new - new[0]
    s = pos[1:] - pos[:-1]
    mid = pos[min(F // 2 + 1, F - 1)]
    fs = -pos + mid
    return {"pair_b": b, "final_shift": s, "frame_shift": fs,
            "sum": _exact_image(_exact_sum(specs, n, fs), n)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "movie":
        return _exact_movie(case, seed)
    if kind == "batch":
        return [_exact_movie(m, seed * 64 + i) for i, m in enumerate(_batch_movies(case))]
    n = case["n"]
    if kind == "pairs":
        s = torch.from_numpy(_spectra(n, case["frames"], seed, case["dose"])).cuda().double()
        s = torch.view_as_complex(s.reshape(case["frames"], n, n // 2 + 1, 2))
        box = _Box(n, case["box"], case["bft"])
        maps = [box(s[i], s[j]) for i, j in _pairs_of(case["frames"], case["fod"])]
        pk = np.array([_exact_peak(m, n) for m in maps])
        return {"b": pk[:, :2], "cc": pk[:, 2], "boxes": torch.stack(maps)}
    if kind == "sharpness":
        F = case["frames"]
        s = torch.from_numpy(_spectra(n, F, seed, case["dose"])).cuda().double()
        s = torch.view_as_complex(s.reshape(F, n, n // 2 + 1, 2))
        t = _drift(F, seed)
        t = -t + np.random.default_rng(seed).normal(0.0, 0.1, t.shape)
        kx, y = _x_index(n)
        w = torch.exp(-0.5 * case["bft"] / n / n * (kx[None, :] ** 2 + y[:, None] ** 2))
        w[:, 1:-1] *= 2
        total = _exact_sum(s, n, t)
        grad = np.empty((F, 2))
        for f in range(F):
            im = (total.conj() * _exact_sum(s[f: f + 1], n, t[f: f + 1])).imag
            v = -2 * w * im * (2 * math.pi / n)
            grad[f] = float((v * kx[None, :]).sum()), float((v * y[:, None]).sum())
        return {"J": float((w * (total.real ** 2 + total.imag ** 2)).sum()), "grad": grad}
    gen = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.poisson(torch.ones(n, n, device="cuda"), generator=gen)
    b = torch.poisson(torch.ones(n, n, device="cuda"), generator=gen)
    spec = torch.view_as_real(torch.fft.rfft2(a.double())).reshape(n, n + 2)
    image = _exact_image(torch.fft.rfft2(b.double()).to(torch.complex64).to(C128), n) * (n * n)
    return {"spectrum": spec, "image": image}
