"""Particle readback returns the caller's order, bit for bit, whatever order the device keeps, for counts
around a workgroup's 256 and for positions or velocities alone."""
import ctypes as C

import numpy as np
import pytest

from banana_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 255, 256, 257, 5000])
def test_readback_user_order(bnn, n):
    params, _ = scenes.dam_break(24)
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    vel = rng.normal(0, 1, (n, 3)).astype(np.float32)
    g = bnn.FLIPSolver(params)
    g.set_particles(pos, vel)
    for _ in range(2):  # as set, then cell-sorted
        p, v = g.particles()
        assert np.array_equal(p, pos) and np.array_equal(v, vel)
        only = np.full_like(pos, -7.0)
        at = only.ctypes.data_as(C.c_void_p)
        g._c(g.L.bnn_flip_get_particles(g.h, at, None))
        assert np.array_equal(only, pos)
        g._c(g.L.bnn_flip_get_particles(g.h, None, at))
        assert np.array_equal(only, vel)
        g.bin_particles()
    g.map_particles_to_grid()  # the readback left the cell-sorted records alone
    h = bnn.FLIPSolver(params)
    h.set_particles(pos, vel)
    h.map_particles_to_grid()
    assert np.array_equal(g.grid("u"), h.grid("u"))
    g.close()
    h.close()
