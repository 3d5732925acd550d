"""The one-launch solve of small grids: every pair of its sides and the sides just outside
it (three launches), one plan's results against numpy's FFT, and in a wake against the
generic kernels.  Tolerance: the 1e-13 the solves are held to elsewhere (about 50 roundings
of 1.1e-16 each); the wakes agree as the two kernel families do elsewhere."""
import itertools

import numpy as np
import pytest

from conftest import rel_err
from test_gpu_lengths import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2", list(itertools.product((32, 48, 64), repeat=2)) + [(16, 64), (64, 96), (31, 64)])
def test_small_solve(qp_ctx, n1, n2):
    from quetzalpic_amd import capi
    f = capi.Fourier2d(qp_ctx, n1, n2)
    for D in (0.0, 10.0, 0.0):
        src = np.random.default_rng(n1 * 100 + n2).standard_normal((n1, n2))
        want = reference(src, 20.0 / n1, 24.0 / n2, D)
        assert rel_err(f.solve_poisson_equation(src, 20.0 / n1, 24.0 / n2, D), want)[0] < 1e-13
    f.close()


@pytest.mark.parametrize("fp64,tol", [(False, 1e-7), (True, 1e-10)])
@pytest.mark.parametrize("ny,nz", [(48, 64), (64, 32)])
def test_small_wake_agrees_with_generic_kernels(qp_ctx, oracle, monkeypatch, ny, nz, fp64, tol):
    """Twelve slices with either family.  The solves differ by 1e-15; on the mixed path that
    flips roundings of positions to 2^-32 of a cell (2e-10 of a particle's deposit, a few of
    them per particle and pass), on the FP64 path the passes amplify it by less than 1e5."""
    from quetzalpic_amd import capi
    fields = ("psi", "ex", "ey", "ez", "by", "bz", "jx")
    g = oracle.grid_from_box(1.2, 20.0, 20.0, 0.1, 20.0 / ny, 20.0 / nz, K=3)
    y, z, w = oracle.init_lattice(g, 2, 2)
    got = []
    for family in ("wave", "generic"):
        monkeypatch.setenv("QP_FFT", family)
        wk = capi.Wake(qp_ctx, g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.ly, g.lz, K=3,
                       precision=capi.QP_PREC_FP64 if fp64 else capi.QP_PREC_MIXED)
        wk.set_particles(y, z, w, np.zeros_like(y), np.zeros_like(y))
        wk.set_laser_gaussian(1.5, 3.0, 6.0, 6.0, 0.8, 10.3, 9.8)
        out, stopped, _ = wk.run(fields=fields)
        assert stopped == 0
        got.append(out)
        wk.close()
    for f in fields:
        assert rel_err(got[0][f], got[1][f])[0] < tol, f
