"""The multigrid preconditioner over hierarchies of every depth and shape its one-workgroup tail takes:
a single brick, two bricks, 2x2x2 bricks, long rows of bricks along each axis, deep cubes.

Bars: M^-1 is symmetric: z1.r2 and z2.r1 differ by the rounding of one FP32 V-cycle, a few hundred
operations a cell (500 2^-24 of sqrt((z1.r1)(z2.r2)), rounded up). The refined solve through it agrees
with the Jacobi-preconditioned one: both reach a residual of 1e-10 max|b|, and the system's condition
number is below 1e4 at these sizes.
"""
import numpy as np
import pytest

from banana_amd import scenes

pytestmark = pytest.mark.gpu

DT = np.float32(1.0 / 600.0)


@pytest.mark.parametrize("cells", [(4, 4, 4), (11, 4, 4), (12, 12, 12), (60, 6, 5), (5, 60, 6), (6, 5, 60), (124, 4, 4), (28, 26, 27), (44, 20, 61)])
def test_mg_tail_shapes(bnn, cells):
    h = 1.0 / 64.0
    params = scenes.base_params(64, boundary_sdf_at_init=True)
    params.update(box_max=tuple(c * h for c in cells), pressure_mode=1, refine_tolerance=1e-10, max_cg_iteration=20000)
    rng = np.random.default_rng(sum(cells))
    n = 6 * cells[0] * cells[1] * cells[2]
    pos = (rng.uniform(0, 1, (n, 3)) * np.array(cells) * [1.0, 0.8, 1.0] * h).astype(np.float32)
    vel = rng.normal(0, 0.5, pos.shape).astype(np.float32)
    out = {}
    for precond in (1, 0):
        g = bnn.FLIPSolver(dict(params, preconditioner=precond))
        g.set_particles(pos, vel)
        g.map_particles_to_grid()
        g.pressure_projection(DT)
        assert g.stats()["pcg_success"] == 1
        out[precond] = g.pressure()
        if precond == 1:
            r = rng.normal(0, 1, (2, out[1].size))
            r[:, out[1] == 0] = 0  # empty rows
            z = [g.apply_preconditioner(v) for v in r]
            zr = [[float(a @ b) for b in r] for a in z]
            assert zr[0][0] > 0 and zr[1][1] > 0
            assert abs(zr[0][1] - zr[1][0]) <= 1e-4 * np.sqrt(zr[0][0] * zr[1][1])
        g.close()
    assert np.linalg.norm(out[1] - out[0]) <= 1e-6 * np.linalg.norm(out[0])


def test_mg_coarsest_of_two_bricks(bnn):
    """An axis of more than 8 * 2^15 cells leaves the coarsest of the 16 levels with more than one brick, which
    the tail does not take: fluid on both sides of the border between its two, and far from it."""
    h = 1.0 / 16.0
    nz = 8 * 2 ** 15 + 10
    params = scenes.base_params(16)
    params.update(box_max=(6 * h, 5 * h, nz * h), pressure_mode=1, refine_tolerance=1e-10, max_cg_iteration=20000)
    rng = np.random.default_rng(5)
    pos = np.concatenate([rng.uniform(0, 1, (8 * 30 * (hi - lo), 3)) * [6 * h, 5 * h, (hi - lo) * h] + [0, 0, lo * h]
                          for lo, hi in ((nz - 30, nz - 1), (100000, 100040), (3, 20))]).astype(np.float32)
    vel = rng.normal(0, 0.5, pos.shape).astype(np.float32)
    out = {}
    for precond in (1, 0):
        g = bnn.FLIPSolver(dict(params, preconditioner=precond))
        assert g.n[2] > 8 * 2 ** 15
        g.set_particles(pos, vel)
        g.map_particles_to_grid()
        g.pressure_projection(DT)
        assert g.stats()["pcg_success"] == 1
        out[precond] = g.pressure()
        if precond == 1:
            r = rng.normal(0, 1, (2, out[1].size))
            r[:, out[1] == 0] = 0  # empty rows
            z = [g.apply_preconditioner(v) for v in r]
            zr = [[float(a @ b) for b in r] for a in z]
            assert zr[0][0] > 0 and zr[1][1] > 0
            assert abs(zr[0][1] - zr[1][0]) <= 1e-4 * np.sqrt(zr[0][0] * zr[1][1])
        g.close()
    assert np.linalg.norm(out[1] - out[0]) <= 1e-6 * np.linalg.norm(out[0])
