"""GPU tests of the cell search of the peak kernel (FindShift,
cufunc.cu:396-497): only the 8 x 8 cells of the 512 x 512 interpolated map
whose bound reaches the best cell centre are evaluated point by point, so maps
where many, one or all cells are kept must give the maximum of the full search.

Noise (the most kept cells), one peak anywhere including the box's edge, a
smooth hill (few distinct values), a peak on a large constant, and the excluded
square around the centre, which may hold the highest points (wnoise >= 0) or
everything.  Shifts identical to the FP64 oracle's full search of the same FP32
map; cc within 1e-9 (both sides FP64, sums of 150 terms)."""
import numpy as np
import pytest

import motioncorr1exp_amd as mc
from _oracle import Oracle

pytestmark = pytest.mark.gpu
N = 512


@pytest.fixture(scope="module")
def o():
    return Oracle("f64")


@pytest.fixture(scope="module")
def ctx():
    c = mc.Context(0)
    yield c
    c.close()


def _maps(kind, box, count):
    rng = np.random.default_rng(box * 7 + len(kind))
    y, x = np.mgrid[0:box, 0:box]
    out = np.empty((count, box, box), np.float32)
    for q in range(count):
        x0, y0 = rng.uniform(-1, box, 2)
        g = lambda s: np.exp(-((x - x0) ** 2 + (y - y0) ** 2) / (2 * s * s))
        out[q] = {"noise": lambda: rng.normal(0, 1.0, (box, box)),
                  "peak": lambda: 50 * g(1.0) + rng.normal(0, 1.0, (box, box)),
                  "hill": lambda: g(5.0) + 1e-4 * rng.normal(0, 1.0, (box, box)),
                  "base": lambda: 1e4 + g(2.0) + 0.3 * rng.normal(0, 1.0, (box, box)),
                  "negative": lambda: -1e3 + rng.normal(0, 1.0, (box, box))}[kind]()
    return out


@pytest.mark.parametrize("wnoise", [-1, 0, 6])
@pytest.mark.parametrize("box", [16, 33, 96])
@pytest.mark.parametrize("kind", ["noise", "peak", "hill", "base", "negative"])
def test_cell_search_matches_full_search(ctx, o, kind, box, wnoise):
    maps = _maps(kind, box, 12)
    b, cc = ctx.find_peaks(maps, N, wnoise)
    for q in range(len(maps)):
        ox, oy, occ = o.find_shift_box(maps[q].astype(np.float64), N, wnoise)
        assert (b[q, 0], b[q, 1]) == (ox, oy), q
        assert abs(cc[q] - occ) <= 1e-9 * abs(occ), q


def test_maps_without_a_maximum(ctx, o):
    """Nothing admitted, a zero map (every point ties) and a NaN in the window:
    the start point U[0], as in the full search."""
    rng = np.random.default_rng(3)
    m = rng.normal(0, 1.0, (1, 32, 32)).astype(np.float32)
    b, cc = ctx.find_peaks(m, N, 64)
    ox, oy, occ = o.find_shift_box(m[0].astype(np.float64), N, 64)
    assert (b[0, 0], b[0, 1]) == (ox, oy) and abs(cc[0] - occ) <= 1e-9 * abs(occ)
    b, cc = ctx.find_peaks(np.zeros((3, 32, 32), np.float32), N)
    assert (b == -16).all() and (cc == 0).all()
    m[0, 3, 5] = np.nan
    m[0, 5, 7] = 100.0
    b, cc = ctx.find_peaks(m, N)
    assert (b[0] == -16).all() and np.isnan(cc[0])


@pytest.mark.parametrize("wnoise", [-1, 3])
@pytest.mark.parametrize("box", [16, 96])
@pytest.mark.parametrize("kind", ["constant", "minus", "stripes", "inf"])
def test_maps_that_keep_most_cells(ctx, o, kind, box, wnoise):
    """Maps without a single maximum: every point ties up to rounding (1e-14 of the
    value), so the value is compared and not the place; one map alone and twelve at
    once give the same bits."""
    y, x = np.mgrid[0:box, 0:box]
    m = {"constant": np.full((box, box), 0.37), "minus": np.full((box, box), -2.5e4),
         "stripes": np.cos(2 * np.pi * (6 * x + 3 * y) / 16), "inf": np.full((box, box), np.inf)}[kind]
    m = np.repeat(m.astype(np.float32)[None], 12, axis=0)
    b, cc = ctx.find_peaks(m, N, wnoise)
    b1, cc1 = ctx.find_peaks(m[:1], N, wnoise)
    assert (b == b1).all() and (cc.view(np.int64) == cc1.view(np.int64)).all()
    if kind == "inf":
        assert np.isnan(cc).all() and (b == -(box // 2)).all()
    else:
        occ = o.find_shift_box(m[0].astype(np.float64), N, wnoise)[2]
        assert abs(cc[0] - occ) <= 1e-9 * abs(occ)
