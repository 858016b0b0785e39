"""GPU tests of the sharpness pass (sum, J and dJ/ds in one pass over the
frames up to 64 frames, after a sum of its own above) against the FP64 oracle:
frame counts at the edges of its forms (one and two frames, odd counts, the last
of each tile width, 64 and 65, several frame blocks), sizes with chunks of less
than a tile and tiles over several columns, and frames left out (NaN shift),
whose gradient is zero.  Spectra of random real images, so J and the gradient
are sums without structure; the only difference from the oracle is the FP32
phase factor and product (about 3e-7 of an element), so J within 2e-6 and the
gradient within 1e-5 of its largest component."""
import numpy as np
import pytest

import motioncorr1exp_amd as mc
from _oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F,skip", [
    (64, 1, ()), (64, 2, ()), (66, 3, (1,)), (128, 4, ()), (96, 5, (0,)), (250, 24, (3, 23)),
    (256, 37, ()), (64, 38, ()), (64, 39, ()), (64, 51, ()), (64, 52, ()), (130, 64, (63,)),
    (64, 65, (0, 64)), (130, 77, ()), (64, 130, (38, 39))])
def test_sum_value_and_gradient_match_oracle(n, F, skip):
    rng = np.random.default_rng(n * 1000 + F)
    spec = np.fft.rfft2(rng.standard_normal((F, n, n))).astype(np.complex64)
    s = rng.normal(0, 2.0, (F, 2))
    s[list(skip)] = np.nan
    ctx = mc.Context(0)
    ctx.set_spectra(spec.view(np.float32))
    J, g = ctx.sharpness(s, 150.0)
    ctx.close()
    keep = [f for f in range(F) if f not in skip]
    oJ, og = Oracle("f64").sharpness(spec[keep].view(np.float32).astype(np.float64), n, 150.0, s[keep])
    print("J", abs(J - oJ) / abs(oJ), "gradient", np.abs(g[keep] - og).max(), np.abs(og).max())
    assert abs(J - oJ) <= 2e-6 * abs(oJ)
    # one frame: Im(conj(S) S) = 0, so the scale is that of the terms, which
    # round S twice (2^-24 each way) and carry a factor of at most 2 pi: 4e-7 J
    scale = 1e-5 * np.abs(og).max() if len(keep) > 1 else 4e-7 * oJ
    assert np.abs(g[keep] - og).max() <= scale
    assert (g[list(skip)] == 0).all()


def test_two_threads_of_different_lds():
    """Contexts on two threads whose sharpness launches need 81 and 36 KB of the same
    kernel's LDS: the values of each alone, bit for bit."""
    import threading

    n, out, alone = 128, {}, {}
    rng = np.random.default_rng(11)
    specs = {F: np.fft.rfft2(rng.normal(0, 1, (F, n, n))).astype(np.complex64) for F in (38, 16)}
    shift = {F: rng.normal(0, 1.5, (F, 2)) for F in specs}

    def run(F, reps, to):
        ctx = mc.Context(0)
        ctx.set_spectra(specs[F].view(np.float32))
        to[F] = [ctx.sharpness(shift[F], 150.0) for _ in range(reps)]
        ctx.close()

    for F in specs:
        run(F, 1, alone)
    threads = [threading.Thread(target=run, args=(F, 40, out)) for F in specs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for F in specs:
        j, g = alone[F][0]
        assert len(out[F]) == 40 and all(a == j and np.array_equal(b, g) for a, b in out[F])
