"""pf_dft's passes at their edges against numpy in FP64: every number of
radix-8 passes and remainders (powers of two), the longest chirp forms of one
block and the first of the four-step path, from real and complex input,
through both entry points.  The bar is 1e-11 of the largest magnitude, as
for the other transform tests."""
import ctypes

import numpy as np
import pytest

from phonomena_amd import fdtd

pytestmark = pytest.mark.gpu


def _close(got, want):
    assert got.shape == want.shape
    assert float(np.max(np.abs(got - want))) <= 1e-11 * float(np.max(np.abs(want)))


@pytest.mark.parametrize("n,nf", [(2 ** e, 2 ** e) for e in range(1, 14)] + [
    (3, 1), (5, 5), (171, 86), (4097, 4096), (4097, 4097),  # n + nf - 1 at 2^13 and one beyond
    (5462, 2731), (8191, 2), (16384, 1), (11000, 5385), (11000, 5386)])
def test_passes_and_convolution_lengths(n, nf):
    rng = np.random.default_rng(n + nf)
    x = rng.standard_normal((3, n))
    z = x + 1j * rng.standard_normal((3, n))
    _close(fdtd.dft(x, nf=nf, scale=0.5), 0.5 * np.fft.fft(x)[:, :nf])
    w = rng.uniform(0.5, 1.0, n)
    want = np.fft.fft(z * w)[:, :nf]
    _close(fdtd.dft(z, nf=nf, window=w), want)
    # the entry point with separate real and imaginary arrays
    re, im = np.ascontiguousarray(z.real), np.ascontiguousarray(z.imag)
    ore, oim = np.empty((3, nf)), np.empty((3, nf))
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    fdtd.check(fdtd.load().pf_dft(vp(re), vp(im), 3, n, nf, vp(w), 1.0, vp(ore), vp(oim)))
    _close(ore + 1j * oim, want)
