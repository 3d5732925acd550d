"""Envelope steps on a device with no room for a pipeline's buffers: the steps run
with what the envelope has, one at a time, and give what single steps give."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class FullDevice:
    """Takes the device's free memory in ever smaller pieces, down to 4 MB."""

    def __enter__(self):
        from quetzalpic_amd import capi
        self.lib, self.held = capi.load(), []
        size = 1 << 36
        while size >= 1 << 22:
            p = ctypes.c_void_p()
            if self.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
                self.held.append(p)
            else:
                size //= 2
        self.lib.hipGetLastError()
        return self

    def __exit__(self, *exc):
        for p in self.held:
            self.lib.hipFree(p)


def test_steps_without_memory_for_a_pipeline(qp_ctx):
    from quetzalpic_amd import capi
    nx, ny, nz, steps = 6, 256, 256, 7
    rng = np.random.default_rng(3)
    chi = 1.0 + 0.3 * rng.random((nx, ny, nz))

    def env():
        e = capi.Envelope(qp_ctx, nx, ny, nz, 0.1, 20.0 / ny, 20.0 / nz, 20.0)
        e.set_gaussian(1.0, 0.4, 6.0, 6.0, 0.3, 10.0, 10.0)
        e.set_chi(chi)
        return e

    ref = env()
    for _ in range(steps):
        ref.advance(2.0, steps=1, chi_iterations=1, use_graph=0)
    got = env()
    with FullDevice() as full:
        assert full.held
        got.advance(2.0, steps=steps, chi_iterations=1, use_graph=0)   # 15 MB of buffers
    assert np.array_equal(got.get(), ref.get())
    got.advance(2.0, steps=steps, chi_iterations=1, use_graph=0)       # with room again
    ref.advance(2.0, steps=steps, chi_iterations=1, use_graph=0)
    assert np.array_equal(got.get(), ref.get())
    got.close()
    ref.close()
