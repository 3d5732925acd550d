"""The push launches share one window per particle block, taken from the block's
cells: grids whose sides the window does not fit, half steps that leave it,
blocks of one, four and nine particles per cell, and passes that stop.

The mixed path is compared with the plain FP64 path (one kernel per loop, no
windows) on the same inputs.  Tolerances: the path's bar of 1e-5 on psi and e_x,
1e-4 on the other fields (as in test_gpu_configs.py)."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

FIELDS = ("psi", "ex", "ey", "by", "bz", "rho", "jx", "jy", "chi")
L = 20.0


def both(qp_ctx, oracle, ny, nz, ppc, dx, nx, a0, K=3, kick=0.0, tile=None, fields=FIELDS, b_threshold=100.0):
    from quetzalpic_amd import capi
    g = oracle.grid_from_box(nx * dx, L, L, dx, L / ny, L / nz, K=K)
    y, z, w = oracle.init_lattice(g, ppc, ppc)
    rng = np.random.default_rng(ny + 7 * nz + ppc)
    py, pz = kick * rng.standard_normal(len(y)), kick * rng.standard_normal(len(y))
    out = []
    for prec in (capi.QP_PREC_FP64, capi.QP_PREC_MIXED):
        wk = capi.Wake(qp_ctx, g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.ly, g.lz, K=K, precision=prec,
                       b_threshold=b_threshold)
        wk.set_particles(y, z, w, py, pz)
        wk.set_laser_gaussian(a0, 3.0, 6.0, 6.0, 0.7 * nx * dx, L / 2, L / 2)
        if prec == capi.QP_PREC_MIXED and tile:
            wk.set_tile(*tile)
        out.append(wk.run(fields=fields))
        wk.close()
    return out


def check(ref, got, fields=FIELDS):
    for f in fields:
        e = rel_err(got[f], ref[f])
        assert e[0] < (1e-5 if f in ("psi", "ex") else 1e-4), (f, e)


@pytest.mark.parametrize("ny,nz", [(16, 16), (18, 20), (19, 33), (40, 24), (64, 48)])
@pytest.mark.parametrize("ppc", [1, 2, 3])
def test_grids_and_particles_per_cell(qp_ctx, oracle, ny, nz, ppc):
    (ref, s0, _), (got, s1, _) = both(qp_ctx, oracle, ny, nz, ppc, 0.1, 12, 1.0)
    assert s0 == s1 == 0
    check(ref, got)


@pytest.mark.parametrize("tile", [(256, 640), (128, 384), (256, 1024)])
def test_half_steps_beyond_the_window(qp_ctx, oracle, tile):
    """dx = 0.5 against cells of 0.3125 and momenta of order 2: many half steps leave
    their block's window (those particles deposit with global atomics)."""
    (ref, s0, _), (got, s1, _) = both(qp_ctx, oracle, 64, 64, 2, 0.5, 6, 0.5, K=2, kick=2.0, tile=tile)
    assert s0 == s1 == 0
    check(ref, got)


@pytest.mark.parametrize("K,thr", [(1, 0.02), (2, 0.02), (3, 0.02), (4, 0.05), (5, 0.01)])
def test_jx_of_a_stopped_pass(qp_ctx, oracle, K, thr):
    """The final view of a stopped pass holds the jx of the iteration that stopped it
    (planes alternate between iterations), on both paths."""
    (ref, s0, i0), (got, s1, i1) = both(qp_ctx, oracle, 32, 32, 2, 0.1, 30, 1.5, K=K, b_threshold=thr)
    assert s0 == s1 == 1 and i0 == i1
    e = rel_err(got["jx"][0], ref["jx"][0])
    assert np.abs(ref["jx"][0]).max() > 0 and e[0] < 1e-4, e
    for f in ("by", "bz", "chi"):
        e = rel_err(got[f][i0], ref[f][i0])
        assert e[0] < 1e-4, (f, e)
