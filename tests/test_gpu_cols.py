"""The pair stage's column pass (mc_cols.hip) at the sizes where it can go
wrong: transform sizes whose share per wave is full, ragged or a fraction of
a wave, one to eight waves per item, every radix of the sizes that are not
multiples of 128 (16, 14, 12, 10, 8, 6; even and odd shares, boxes of one to
three tiles), boxes from 16 to the largest, odd ones and both sides of 96
among them.  Box maps of random spectra set directly,
against the FP64 cross power and inverse of the same spectra by numpy
(cufunc.cu:343-370, DFAlign.cu:897, cufunc.cu:398-407).

Bound: the map is a sum of n^2/2 products by FP32 transforms of length n and
a sum over n/2 bins, whose rounding errors add as random terms: about
2^-24 sqrt(2 log2 n + 2) of the map's root mean square per point for the
transforms and as much again for the sum, 7e-7 at n = 8192 with peaks of five
standard deviations; 2e-6 of the map's maximum holds all of it."""
import numpy as np
import pytest

import motioncorr1exp_amd as mc

pytestmark = pytest.mark.gpu


def reference_box(a, b, n, bfactor, box):
    """Central box of irfft2(a conj(b) z) / normalisation in FP64 (rows by FFT,
    box columns by direct sums)."""
    kx = np.arange(n // 2 + 1)
    y = np.where(np.arange(n) < n // 2, np.arange(n), np.arange(n) - n)
    m = -0.5 * bfactor / n / n
    z = np.exp(m * (kx[None, :] ** 2 + y[:, None] ** 2)) * (1 - 2 * ((kx[None, :] + y[:, None]) % 2))
    o = (n - box) // 2
    t = np.fft.ifft(a * np.conj(b) * z / (n * (n // 2 + 1)), axis=0, norm="forward")[o:o + box]
    w = np.full(n // 2 + 1, 2.0)
    w[0] = w[-1] = 1.0
    e = np.exp(2j * np.pi * ((kx[:, None] * (o + np.arange(box))[None, :]) % n) / n)
    return ((t * w) @ e).real


@pytest.fixture(scope="module")
def ctx():
    c = mc.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,box", [
    (128, 16), (128, 128), (256, 96), (256, 127), (512, 33), (512, 96), (512, 128), (768, 95),
    (1024, 64), (1024, 97), (1280, 96), (1280, 126), (1536, 17), (1920, 96), (2048, 96),
    (2560, 128), (3072, 70), (3840, 96), (3840, 128), (4096, 96), (5120, 96), (6144, 111),
    (8192, 96), (8192, 128),
    # radix 16, 14, 12, 10, 8, 6 (and 4096 with a box above 128)
    (64, 33), (64, 64), (1808, 96), (1808, 129), (4096, 200), (512, 256),
    (70, 64), (1022, 96), (3710, 96), (3710, 113), (3710, 224),
    (132, 96), (4092, 96), (4092, 97), (4092, 192),
    (110, 80), (2470, 96), (2470, 81), (2470, 160),
    (72, 64), (1000, 65), (2472, 96), (2472, 192), (4024, 128),
    (66, 48), (102, 49), (1854, 96), (1854, 97), (2046, 144), (4098, 96)])
def test_box_maps_match_fp64(ctx, n, box):
    F = 3
    rng = np.random.default_rng(n + box)
    spec = np.fft.rfft2(rng.standard_normal((F, n, n))).astype(np.complex64)
    ctx.set_spectra(spec.view(np.float32))
    pairs = np.array([(0, 1), (0, 2), (2, 1), (1, 1)], np.int32)
    _, _, maps = ctx.pair_shifts(pairs, 150.0, box, want_boxes=True)
    worst = 0.0
    for q, (a, b) in enumerate(pairs):
        ref = reference_box(spec[a].astype(np.complex128), spec[b].astype(np.complex128), n, 150.0, box)
        worst = max(worst, float(np.abs(maps[q] - ref).max() / np.abs(ref).max()))
    print("n %d box %d: max error / max %.3g" % (n, box, worst), flush=True)
    assert worst < 2e-6


@pytest.mark.parametrize("n,box", [(5766, 128), (7672, 144), (8170, 80), (8184, 129), (8184, 192)])
def test_many_waves_and_tiles(ctx, n, box):
    """Three tiles of 16 waves exceed the LDS and take the chirp-z pass (5766,
    8184); 15 waves of three tiles (7672) and 13 of a wide exchange (8170) fit.
    Two white spectra, one pair; reference and bound as above."""
    rng = np.random.default_rng(n + box)
    spec = rng.standard_normal((2, n, n + 2), np.float32)
    ctx.set_spectra(spec)
    _, _, maps = ctx.pair_shifts(np.array([(0, 1)], np.int32), 150.0, box, want_boxes=True)
    a, b = spec.view(np.complex64)
    ref = reference_box(a.astype(np.complex128), b.astype(np.complex128), n, 150.0, box)
    worst = float(np.abs(maps[0] - ref).max() / np.abs(ref).max())
    print("n %d box %d: max error / max %.3g" % (n, box, worst), flush=True)
    assert worst < 2e-6


def test_more_waves_after_fewer(ctx):
    """One kernel at eight waves (80 KB of LDS), one wave (10 KB) and eight again:
    the map of the first call, bit for bit."""
    got = []
    for n in (8192, 128, 8192):
        spec = np.random.default_rng(n).standard_normal((2, n, n + 2), np.float32)
        ctx.set_spectra(spec)
        got.append(ctx.pair_shifts(np.array([(0, 1)], np.int32), 150.0, 96, want_boxes=True)[2])
    assert np.array_equal(got[0], got[2])


@pytest.mark.parametrize("n,box", [(384, 129), (384, 200), (1152, 256), (1920, 160)])
def test_large_boxes_at_odd_multiples_of_128(ctx, n, box):
    """Boxes above 128 at sizes that are a multiple of 128 and not of 256: the rows
    start at n/2 - 128, a multiple of 64 there too."""
    test_box_maps_match_fp64(ctx, n, box)
