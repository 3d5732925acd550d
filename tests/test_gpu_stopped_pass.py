"""Passes that stop (|B| over the threshold): what they leave, and that they end there.

A pass without a callback learns from the device that its members have stopped and
enqueues at most two watch periods of eight slices more.  Tolerances: the mixed
path's bar of 1e-4 on the source planes against FP64 (as in test_gpu_configs.py);
two runs of one path differ by the order of their atomic sums, which can move a
stored position by its 2^-32 of a cell (1.5e-10 here) a slice: 2e-8 in 100 slices."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

L, N, NX, DX = 20.0, 32, 100, 0.1
WATCH = 8
SAME = 2e-8


def grid(oracle, K):
    return oracle.grid_from_box(NX * DX, L, L, DX, L / N, L / N, K=K)


def laser(a0, dx=0.0):
    return (a0, 3.0, 6.0, 6.0, NX * DX - 2.0 - dx, L / 2, L / 2)


def wake(qp_ctx, oracle, K, prec, thr, a0=1.5):
    from quetzalpic_amd import capi
    g = grid(oracle, K)
    y, z, w = oracle.init_lattice(g, 2, 2)
    wk = capi.Wake(qp_ctx, g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.ly, g.lz, K=K, precision=prec, b_threshold=thr)
    wk.set_particles(y, z, w)
    wk.set_laser_gaussian(*laser(a0))
    return wk


@pytest.mark.parametrize("prec,cls,per_iteration", [("FP64", "solve", 2), ("MIXED", "push_B", 1)])
def test_pass_without_callback_ends_where_it_stops(qp_ctx, oracle, prec, cls, per_iteration):
    from quetzalpic_amd import capi
    K = 2
    wk = wake(qp_ctx, oracle, K, getattr(capi, "QP_PREC_" + prec), 0.02)
    _, st, stop = wk.run(fields=("by",))
    want = wk.get_particles()
    ran = NX - stop
    assert st == 1 and 0 < ran < NX // 2
    _, st, stop2 = wk.run()
    assert (st, stop2) == (1, stop)
    for a, b in zip(wk.get_particles(), want):
        assert np.abs(a - b).max() < SAME
    launches, _ = wk.profile_kernel(cls)
    # one psi solve a slice beside the iterations' psi_middle and B solves
    extra = 1 if cls == "solve" else 0
    assert launches <= (ran + 2 * WATCH) * (K * per_iteration + extra), (launches, ran)
    wk.close()


def members(qp_ctx, oracle, n, a0s, K, thr):
    from quetzalpic_amd import capi
    g = oracle.grid_from_box(NX * DX, L, L, DX, L / n, L / n, K=K)
    y, z, w = oracle.init_lattice(g, 2, 2)
    b = capi.WakeBatch(qp_ctx, len(a0s), g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.ly, g.lz, K=K, b_threshold=thr)
    for m, a0 in enumerate(a0s):
        b.set_particles(m, y, z, w)
        b.set_laser_gaussian(m, *laser(a0, 0.5 * m))
    return b


@pytest.mark.parametrize("a0s", [(1.5, 1.5, 1.2), (1.5, 0.02, 1.2), (0.02, 0.01, 0.02)],
                         ids=["all stop", "one runs on", "none stops"])
def test_members_that_stop_at_their_own_slices(qp_ctx, oracle, a0s):
    """Batch and group, with and without a callback: the same stop slices and particles."""
    from quetzalpic_amd import capi
    b = members(qp_ctx, oracle, 32, a0s, 2, 0.02)
    _, _, stops = b.run(fields=("by",))
    want = [b.get_particles(m) for m in range(3)]
    assert [s >= 0 for s in stops] == [a > 0.1 for a in a0s]
    c = members(qp_ctx, oracle, 48, a0s, 2, 0.02)
    _, _, stops_c = c.run(fields=("by",))
    want_c = [c.get_particles(m) for m in range(3)]
    for _ in range(3):   # the later runs replay captured steps
        b.run()
        got = [b.get_particles(m) for m in range(3)]
        assert list(b.run()[2]) == list(stops)
        for x, y in zip(got, want):
            assert max(np.abs(p - q).max() for p, q in zip(x, y)) < SAME
    g = capi.WakeGroup(qp_ctx, [b, c])
    for _ in range(3):
        g.run()
        for h, w in ((b, want), (c, want_c)):
            for m in range(3):
                assert max(np.abs(p - q).max() for p, q in zip(h.get_particles(m), w[m])) < SAME
    g.close()
    c.close()
    b.close()


@pytest.mark.parametrize("K,thr", [(1, 0.02), (2, 0.02), (5, 0.01)])
def test_rho_of_the_final_view(qp_ctx, oracle, K, thr):
    """rho of a stopped pass's final view: the step's own after its last iteration, else
    the slice's before it (the mixed path deposits rho in the last iteration only)."""
    from quetzalpic_amd import capi
    res = []
    for prec in (capi.QP_PREC_FP64, capi.QP_PREC_MIXED):
        wk = wake(qp_ctx, oracle, K, prec, thr)
        res.append(wk.run(fields=("rho",)))
        wk.close()
    (ref, s0, i0), (got, s1, i1) = res
    assert s0 == s1 == 1 and i0 == i1 and i0 < NX - 1
    own, before = rel_err(got["rho"][0], ref["rho"][0])[0], rel_err(got["rho"][0], ref["rho"][i0 + 1])[0]
    assert (own if K == 1 else min(own, before)) < 1e-4, (own, before)
