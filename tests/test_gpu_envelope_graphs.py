"""Envelope calls of changing step counts on one handle: the captured pipelines of
several depths stay side by side, through the growth of the pipeline's buffers and the
steps that an attached wake takes."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def envelope(qp_ctx, nx, ny, nz, seed=1):
    from quetzalpic_amd import capi
    rng = np.random.default_rng(seed)
    e = capi.Envelope(qp_ctx, nx, ny, nz, 0.1, 20.0 / ny, 20.0 / nz, 10.0)
    e.set(rng.standard_normal((nx, ny, nz)) + 1j * rng.standard_normal((nx, ny, nz)))
    e.set_chi(1.0 + 0.5 * rng.random((nx, ny, nz)))
    return e


@pytest.mark.parametrize("ny,nz", [(32, 32), (24, 20)])
def test_changing_step_counts_equal_single_steps(qp_ctx, ny, nz):
    """1, 3, 16, 2, 19 (10 + 9), 5, 7 steps a call, four rounds (direct, captured, replayed,
    depths beyond the graphs held), another dtau in between."""
    e, ref = envelope(qp_ctx, 5, ny, nz), envelope(qp_ctx, 5, ny, nz)
    for rnd in range(4):
        for steps in (1, 3, 16, 2, 19, 5, 7):
            dtau = 0.25 if (rnd, steps) == (2, 2) else 0.5
            e.advance(dtau, steps=steps, chi_iterations=1, use_graph=1)
            for _ in range(steps):
                ref.advance(dtau, steps=1, chi_iterations=1, use_graph=0)
            assert np.array_equal(e.get(), ref.get()), (rnd, steps)
    e.close()
    ref.close()


def test_steps_of_an_attached_wake_between_calls(qp_ctx, oracle):
    """A wake's pass steps the envelope (one step) between calls of three steps; graphs
    against direct launches."""
    from quetzalpic_amd import capi
    g = oracle.grid_from_box(0.8, 20.0, 20.0, 0.1, 20.0 / 32, 20.0 / 32, K=2)
    y, z, w = oracle.init_lattice(g, 1, 1)
    got = []
    for use_graph in (1, 0):
        e = capi.Envelope(qp_ctx, g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, 10.0)
        e.set_gaussian(0.5, 1.0, 6.0, 6.0, 0.5, 10.0, 10.0)
        wk = capi.Wake(qp_ctx, g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.ly, g.lz, K=2, precision=capi.QP_PREC_FP64,
                       use_graph=use_graph)
        wk.set_particles(y, z, w)
        wk.attach_envelope(e)
        wk.set_envelope_step(0.5, 1)
        for _ in range(4):
            wk.run()
            e.advance(0.5, steps=3, chi_iterations=1, use_graph=use_graph)
        got.append(e.get())
        wk.close()
        e.close()
    # the wake's deposits are atomic sums: equal to rounding
    assert np.abs(got[0] - got[1]).max() < 1e-9 * np.abs(got[1]).max()


def test_alternating_step_counts_are_not_captured_anew(qp_ctx):
    """One step, then twelve, by turns: no slower than each repeated by itself (with one
    graph for all, captured anew at each change, 1.6 to 2.2 times)."""
    e = envelope(qp_ctx, 60, 128, 128)

    def best(calls):
        def once():
            t = time.perf_counter()
            for steps in calls:
                e.advance(0.5, steps=steps, chi_iterations=1, use_graph=1)
            return time.perf_counter() - t
        for _ in range(3):
            once()
        return min(once() for _ in range(7))

    apart = best((1,)) + best((12,))
    turns = best((1, 12))
    assert turns < 1.5 * apart, (turns, apart)
    e.close()
