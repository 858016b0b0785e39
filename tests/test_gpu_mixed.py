"""GPU tests of the mixed-factor transforms (mc_mixed.hip), which serve stage 1
and the sum image at sizes without a Stockham plan.

- Forward and inverse 2-D transforms against numpy in FP64 over the forms that
  the factors take: one matrix level (17 to 127), two of them with the last one
  a matrix level too, three and four register levels, every register radix from
  9 to 16, odd and even last factors, rows and columns of different kinds (a
  prime above 127 in one only goes to the chirp-z transform), the sizes at which
  the workgroups change and the largest.  Random data: the transforms' FP32 error
  is a few 1e-7 of the largest output, as for the other transforms.
- Frames of every type with dark and gain, of widths and region origins that
  leave the four-pixel loads misaligned and a remainder, cropped, binned and
  padded: the spectra against numpy on the corrected frames."""
import numpy as np
import pytest

import motioncorr1exp_amd as mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [
    68, 74, 90, 130, 254, 262, 266, 508, 570, 1014, 1170, 1210, 1898, 2002, 2294, 2312, 2890, 3798,
    3802, 4050, 4900, 5000, 6254, 7920, 8188])
def test_forward_and_inverse_against_numpy(n):
    rng = np.random.default_rng(n)
    img = rng.standard_normal((n, n)).astype(np.float32)
    buf = np.zeros((n, n + 2), np.float32)
    buf[:, :n] = img
    d = mc.DeviceArray(buf)
    L = mc.lib()
    plan, iplan = mc.ctypes.c_void_p(), mc.ctypes.c_void_p()
    mc.check(L.mc_fft_plan(mc.ctypes.byref(plan), n))
    mc.check(L.mc_ifft_plan(mc.ctypes.byref(iplan), n))
    mc.check(L.mc_fft2d(d.ptr, plan))
    mc.check(L.mc_sync())
    spec = d.to_host(np.float32, (n, n + 2)).view(np.complex64)
    ref = np.fft.rfft2(img.astype(np.float64))
    err = np.abs(spec - ref).max() / np.abs(ref).max()
    mc.check(L.mc_ifft2d(d.ptr, iplan))
    mc.check(L.mc_sync())
    back = d.to_host(np.float32, (n, n + 2))[:, :n] / (n * n)
    berr = np.abs(back - img).max() / np.abs(img).max()
    L.mc_fft_destroy(plan)
    L.mc_fft_destroy(iplan)
    d.free()
    print("n %d: forward %.3g, round trip %.3g" % (n, err, berr), flush=True)
    assert err <= 1e-6 and berr <= 2e-6


def _spectra(img, nu, n, fill):
    """rfft2 of the images on an nu canvas (rest: the image mean, or none), cropped to n."""
    out = []
    for a in img.astype(np.float64):
        c = np.full((nu, nu), a.mean() if fill else 0.0)
        c[:a.shape[0], :a.shape[1]] = a
        f = np.fft.rfft2(c)[:, :n // 2 + 1]
        out.append(np.concatenate([f[:n // 2], f[nu - n // 2:]]))
    return np.array(out)


@pytest.mark.parametrize("dtype", [np.int8, np.uint8, np.int16, np.uint16, np.float32])
@pytest.mark.parametrize("nx,ny,kw,nu,n", [
    (1001, 799, dict(crop_offsetx=3, crop_offsety=1, crop_nsam=762), 762, 762),  # odd width and origin
    (903, 871, dict(pad=1000), 1000, 1000),                                      # fill, a remainder of 3
    (1115, 1130, dict(crop_nsam=1112, bin=2.0), 1112, 556),                      # Fourier crop
    (345, 333, dict(pad=348), 348, 348)])                                        # rows of 6 x 29
def test_corrected_frames_of_every_type(dtype, nx, ny, kw, nu, n):
    rng = np.random.default_rng(nx)
    F = 3
    frames = rng.poisson(40.0, (F, ny, nx)).astype(dtype)
    dark = rng.normal(2.0, 0.5, (ny, nx)).astype(np.float32)
    gain = rng.normal(1.0, 0.1, (ny, nx)).astype(np.float32)
    host = (frames.astype(np.float32) - dark) * gain
    ctx = mc.Context(0)
    p = mc.default_params(F, FrameDistOffset=1, **kw)
    refs = [mc.DeviceArray(dark), mc.DeviceArray(gain)]
    d, h = mc.DeviceArray(frames), mc.DeviceArray(host)
    ctx.load_frames(d, frames.shape, frames.dtype, p, corr=mc.corrections(*refs))
    got = ctx.get_spectra(F, n)
    ctx.load_frames(h, host.shape, host.dtype, p)
    assert np.array_equal(got, ctx.get_spectra(F, n))
    ctx.close()
    for a in refs + [d, h]:
        a.free()
    ox, oy = kw.get("crop_offsetx", 0), kw.get("crop_offsety", 0)
    region = host if "pad" in kw else host[:, oy:oy + nu, ox:ox + nu]
    ref = _spectra(region, nu, n, "pad" in kw)
    spec = got.view(np.complex64)
    err = np.abs(spec - ref).max() / np.abs(ref).max()
    print("%s %s: %.3g" % (np.dtype(dtype).name, kw, err), flush=True)
    assert err <= 1e-6


@pytest.mark.parametrize("n,F", [(142, 2), (142, 32), (402, 2), (402, 10), (762, 2), (762, 5), (1010, 3)])
def test_frames_on_both_sides_of_the_choice(n, F):
    """Sizes with a large factor, which few frames take through the chirp-z
    transform and many through mixed factors (mc_mixed_form.h)."""
    rng = np.random.default_rng(n + F)
    img = rng.standard_normal((F, n, n), np.float32)
    c = mc.Context(0)
    d = mc.DeviceArray(img)
    c.load_frames(d, img.shape, np.float32, mc.default_params(F))
    got = np.asarray(c.get_spectra(F, n)).view(np.complex64).reshape(F, n, n // 2 + 1)
    c.close()
    d.free()
    ref = np.fft.rfft2(img.astype(np.float64))
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print("n %d, %d frames: %.3g" % (n, F, err), flush=True)
    assert err <= 1e-6
