"""Transform lengths of the generic kernels: every radix of the plan (8, 4, 6, 2, 5,
7, 3, larger primes), blocks of one and of several wavefronts, odd rows, the smallest
and largest sides, against numpy's FFT.  Tolerance: the 1e-13 the solves are held to
elsewhere; a direct sum over a prime of ~1000 terms adds up to sqrt(1000) roundings of
1.1e-16 each per stage, 4e-15."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 13, 20, 21, 26, 35, 36, 49, 50, 55, 63, 65, 77, 100, 120, 121, 125, 127,
           129, 160, 200, 210, 250, 255, 257, 300, 317, 343, 360, 400, 500, 513, 600, 625, 729, 770, 800, 1000, 1009,
           1020, 1021, 1022, 1023]


def reference(src, d1, d2, D):
    n1, n2 = src.shape
    lam = (-D + ((2 * np.cos(2 * np.pi * np.arange(n1) / n1) - 2) / d1 ** 2)[:, None] +
           ((2 * np.cos(2 * np.pi * np.arange(n2 // 2 + 1) / n2) - 2) / d2 ** 2)[None, :])
    lam[0, 0] = 1.0
    f = np.fft.rfft2(src) / lam
    f[0, 0] = 0.0
    return np.fft.irfft2(f, s=src.shape) * (n1 * n2)


@pytest.mark.parametrize("n", LENGTHS)
def test_rows_and_columns_of_a_length(qp_ctx, n):
    from quetzalpic_amd import capi
    for n1, n2, D in ((n, 33, 10.0), (31, n, 0.0)):
        src = np.random.default_rng(n1 * 2000 + n2).standard_normal((n1, n2))
        f = capi.Fourier2d(qp_ctx, n1, n2)
        want = reference(src, 20.0 / n1, 24.0 / n2, D)
        assert rel_err(f.solve_poisson_equation(src, 20.0 / n1, 24.0 / n2, D), want)[0] < 1e-13
        spec = np.fft.rfft2(src)
        assert rel_err(f.forward_transform(src), spec)[0] < 1e-13
        assert rel_err(f.backward_transform(spec), src * (n1 * n2))[0] < 1e-13
        f.close()


@pytest.mark.parametrize("ny,nz", [(25, 30), (100, 21), (200, 120), (1000, 10), (1021, 7)])
def test_envelope_on_generic_lengths(qp_ctx, ny, nz):
    """The envelope's column kernel holds both spectra of a column (two transforms per block)."""
    from oracle import envelope as envo
    from quetzalpic_amd import capi
    nx, dx, dy, dz, k0 = 3, 0.1, 20.0 / ny, 20.0 / nz, 10.0
    rng = np.random.default_rng(ny + nz)
    a = rng.standard_normal((nx, ny, nz)) + 1j * rng.standard_normal((nx, ny, nz))
    chi = 1.0 + 0.5 * rng.random((nx, ny, nz))
    env = capi.Envelope(qp_ctx, nx, ny, nz, dx, dy, dz, k0)
    env.set(a)
    env.set_chi(chi)
    env.advance(0.5, steps=2, chi_iterations=1)
    got = env.get()
    env.close()
    want = envo.advance(a, chi, 0.5, k0, dx, dy, dz, steps=2, m=1)
    assert np.abs(got - want).max() < 1e-11 * np.abs(want).max()
