"""Extrapolation from arbitrary valid flags, bit for bit against the oracle: scattered faces (a layer of
a brick then has more faces to fill than its list holds), a few lone ones, solid blocks, and flags up
to the array's edges, on grids whose rows end at every offset of a 4-face load.
"""
import numpy as np
import pytest

from banana_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(12, 9, 10), (13, 17, 12), (6, 24, 19), (23, 7, 8)])
@pytest.mark.parametrize("density", [0.0, 0.002, 0.06, 0.5, 1.0])
def test_extrapolate_any_flags(oracle, bnn, cells, density):
    h = 1.0 / 16.0
    params = scenes.base_params(16)
    params.update(box_max=tuple(c * h for c in cells))
    g, o = bnn.FLIPSolver(params), oracle.Oracle(params)
    rng = np.random.default_rng(sum(cells) + int(1000 * density))
    faces = (("u", oracle.F_U, oracle.F_VALID_U, oracle.F_EXTRAP_U), ("v", oracle.F_V, oracle.F_VALID_V, oracle.F_EXTRAP_V),
             ("w", oracle.F_W, oracle.F_VALID_W, oracle.F_EXTRAP_W))
    for c, f, fv, _ in faces:
        shape = g.field_shape(c)
        valid = (rng.uniform(size=shape) < density).astype(np.int8)
        if 0.0 < density < 0.5:  # and a solid block
            valid[: shape[0] // 3, shape[1] // 2:, : shape[2] // 2] = 1
        vel = np.where(valid, rng.normal(0, 1, shape), 0).astype(np.float32)
        g.set_grid(c, vel)
        g.set_grid("valid_" + c, valid)
        o.set_field(f, vel)
        o.set_field(fv, valid)
    for _ in range(2):
        g.extrapolate_velocity()
        o.extrapolate_velocity()
        for c, f, fv, fe in faces:
            assert np.array_equal(g.grid(c), o.field(f).astype(np.float32)), c
            assert np.array_equal(g.grid("valid_" + c), o.field(fv)), c
            assert np.array_equal(g.grid("extrap_" + c), o.field(fe)), c
    g.close()
