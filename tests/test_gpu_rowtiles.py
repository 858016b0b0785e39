"""GPU test of the pair row pass over its tiles: boxes at the edges of the row and
column blocks (one block and the first of the next, up to 256), odd boxes (whose
centre column has no mirror), and bin ranges of waves that hold one, few or no
whole step of four bins.  Spectra of random real images; the reference is the box
of the full inverse transform of the weighted cross power in FP64 (the weights of
cufunc.cu:309-341 by the oracle).  FP32 sums of n^2/2 terms through two passes:
2e-6 of the largest value, as for the column pass."""
import numpy as np
import pytest

import motioncorr1exp_amd as mc
from _oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box", [
    (64, 16), (64, 31), (64, 64), (66, 33), (130, 65), (256, 95), (256, 96), (256, 97), (512, 127),
    (512, 128), (512, 129), (512, 192), (512, 193), (512, 256), (1024, 47), (1022, 255), (2048, 64)])
def test_box_maps_match_fp64(n, box):
    o = Oracle("f64")
    rng = np.random.default_rng(n * 300 + box)
    spec = np.fft.rfft2(rng.standard_normal((3, n, n))).astype(np.complex64)
    ctx = mc.Context(0)
    ctx.set_spectra(spec.view(np.float32))
    pairs = np.array([(0, 1), (2, 0), (1, 2)], np.int32)
    _, _, boxes = ctx.pair_shifts(pairs, 150.0, box, want_boxes=True)
    ctx.close()
    for q, (a, b) in enumerate(pairs):
        ref = o.pruned_box(o.cross_power(spec[a], spec[b], n, 150.0), box)
        err = np.abs(boxes[q] - ref).max() / np.abs(ref).max()
        print("n %d box %d pair %d: %.3g" % (n, box, q, err), flush=True)
        assert err <= 2e-6
