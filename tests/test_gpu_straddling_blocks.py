"""Particle blocks that straddle two 16 x 16-cell tiles, as re-binned blocks, ragged
grids and density ramps have them: their cell window (17 x 33 or 18 x 33 nodes) fits
the 640 nodes of the default tile, the one with a margin (19 x 35, 20 x 36) does not.
They keep the window, and the fields stay those of the FP64 path.

Tolerances: the mixed path's bar of 1e-5 on psi and e_x, 1e-4 on the other fields
(as in test_gpu_configs.py)."""
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

FIELDS = ("psi", "ex", "ey", "by", "bz", "rho", "jx", "jy", "chi")
L, N = 20.0, 64


@pytest.mark.parametrize("resort_every", [0, 2])
@pytest.mark.parametrize("gap", [16, 100, 250])
def test_straddling_blocks_keep_their_window(qp_ctx, oracle, gap, resort_every):
    from quetzalpic_amd import capi
    g = oracle.grid_from_box(0.4, L, L, 0.05, L / N, L / N, K=2)
    y, z, w = oracle.init_lattice(g, 1, 1)
    # one particle per cell, 256 per tile, one block each; `gap` cells of the first tile
    # empty: every block then ends that many particles inside the next tile
    empty = (y < 16 * L / N) & (z < 16 * L / N) & (16 * (y * N / L).astype(int) + (z * N / L).astype(int) < gap)
    y, z, w = y[~empty], z[~empty], w[~empty]
    assert len(y) == N * N - gap
    out = []
    for prec in (capi.QP_PREC_FP64, capi.QP_PREC_MIXED):
        mixed = prec == capi.QP_PREC_MIXED
        wk = capi.Wake(qp_ctx, g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.ly, g.lz, K=2, precision=prec,
                       resort_every=resort_every if mixed else 0)
        wk.set_particles(y, z, w)
        wk.set_laser_gaussian(0.5, 3.0, 6.0, 6.0, 0.3, L / 2, L / 2)
        if mixed:
            wk.set_tile(256, 640)
        out.append(wk.run(fields=FIELDS))
        if mixed:
            ovf, tot = wk.window_stats()
            assert tot > 0 and ovf == 0, (ovf, tot)
        wk.close()
    (ref, s0, _), (got, s1, _) = out
    assert s0 == s1 == 0
    for f in FIELDS:
        e = rel_err(got[f], ref[f])
        assert e[0] < (1e-5 if f in ("psi", "ex") else 1e-4), (f, e)
