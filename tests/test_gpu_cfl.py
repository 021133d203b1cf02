"""The CFL timestep is dx over the largest |velocity|, wherever on the faces it stands: the first and the
last face of each component, and face counts of every remainder that the four-wide reads leave.

Exact: a maximum rounds nothing, and the quotient is one FP32 division.
"""
import numpy as np
import pytest

from banana_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(4, 4, 4), (5, 4, 6), (5, 5, 5), (7, 9, 5), (64, 33, 41)])
def test_cfl_finds_every_face(bnn, cells):
    h = np.float32(1.0 / 64.0)
    params = scenes.base_params(64)
    params.update(box_max=tuple(c * float(h) for c in cells), min_timestep=1e-9, max_timestep=1e9, cfl_factor=1.0)
    g = bnn.FLIPSolver(params)
    zero = {c: np.zeros(g.field_shape(c), np.float32) for c in "uvw"}
    rng = np.random.default_rng(sum(cells))
    for c in "uvw":
        n = zero[c].size
        for at in (0, 1, n // 2, n - 4, n - 3, n - 2, n - 1):
            vel = {k: rng.uniform(-1, 1, a.shape).astype(np.float32) for k, a in zero.items()}
            vel[c].reshape(-1)[at] = -37.5
            for k, a in vel.items():
                g.set_grid(k, a)
            assert np.float32(g.timestep_cfl()) == np.float32(g.dx) / np.float32(37.5)
    for k, a in zero.items():
        g.set_grid(k, a)
    assert np.float32(g.timestep_cfl()) == np.float32(1e9)
    g.close()
