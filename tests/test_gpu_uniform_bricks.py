"""The pressure solve over bricks whose 512 rows are all the same, above and below the system size at
which such rows are taken from a constant: a cavity with air pockets, so that uniform bricks, bricks cut
by the free surface and wall bricks are neighbours.

Bars: the pressure solves the system rebuilt on the host from phi and the face weights in FP64 to the
solver's own tolerance. The host's sums differ from the device's by their rounding, 8 terms of at most
12 max|A p| 2^-53 each, which the factor 1.01 covers (max|p| dt stays below 1e4 max|b| at these sizes).
"""
import numpy as np
import pytest

from banana_amd import scenes
from banana_amd.serving import Batch
from test_gpu_configs import host_residual

pytestmark = pytest.mark.gpu

DT = np.float32(1.0 / 600.0)


@pytest.mark.parametrize("precond", [1, 0])
@pytest.mark.parametrize("cells", [(80, 80, 80), (72, 72, 72), (136, 60, 90)])
def test_uniform_rows(bnn, cells, precond):
    h = 1.0 / 64.0
    params = scenes.base_params(64, boundary_sdf_at_init=True)
    params.update(box_max=tuple(c * h for c in cells), pressure_mode=1, refine_tolerance=1e-8, max_cg_iteration=20000,
                  preconditioner=precond)
    ax = [(np.arange(2 * c, dtype=np.float32) + 0.5) * np.float32(h / 2) for c in cells]
    pos = np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    size = np.array(cells, np.float32) * np.float32(h)
    for centre, radius in (((0.5, 1.0, 0.5), 0.3), ((0.3, 0.4, 0.7), 0.1)):
        pos = pos[np.linalg.norm(pos / size - np.float32(centre), axis=1) > radius]
    vel = np.random.default_rng(sum(cells)).normal(0, 0.5, pos.shape).astype(np.float32)
    g = bnn.FLIPSolver(params)
    g.set_particles(pos, vel)
    g.map_particles_to_grid()
    g.pressure_projection(DT)
    assert g.stats()["pcg_success"] == 1
    phi = g.grid("phi")
    rmax, bmax, _ = host_residual(phi, g.grid("weight_u"), g.grid("weight_v"), g.grid("weight_w"), g.pressure(), g.rhs(), DT)
    g.close()
    assert bmax > 0 and rmax <= 1.01e-8 * bmax


@pytest.mark.parametrize("dt", [0.0, -1.0 / 600.0])
def test_uniform_rows_without_a_positive_diagonal(bnn, dt):
    """A projection is given its time step as it is: with none or a negative one no row has a positive
    diagonal, so every inverse is 0, the preconditioner gives zeros and the pressure stays 0, on uniform
    bricks as on others."""
    h = 1.0 / 64.0
    params = scenes.base_params(64)
    params.update(box_max=(80 * h,) * 3, max_cg_iteration=50)
    pos = np.stack(np.meshgrid(*[(np.arange(80, dtype=np.float32) + 0.5) * np.float32(h)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = bnn.FLIPSolver(params)
    g.set_particles(pos, np.random.default_rng(1).normal(0, 0.5, pos.shape).astype(np.float32))
    g.map_particles_to_grid()
    g.pressure_projection(np.float32(dt))
    p = g.pressure()
    z = g.apply_preconditioner(np.random.default_rng(2).normal(0, 1, p.size))
    assert g.stats()["pcg_success"] == 0
    g.close()
    assert np.all(p == 0) and np.all(z == 0)


@pytest.mark.parametrize("refined", [0, 1], ids=["fp32", "refined"])
def test_uniform_rows_in_a_batch(bnn, refined):
    """Scenes on both sides of the system size at which the uniform rows' constant is used (1331, 1000 and 1890
    bricks of a full box) in one batch: every bit of the velocities and the pressure is that of the scene alone."""
    h = 1.0 / 64.0
    made = []
    for cells in ((84, 84, 84), (76, 76, 76), (140, 68, 100)):
        params = scenes.base_params(64, boundary_sdf_at_init=True)
        params.update(box_max=tuple(c * h for c in cells), pressure_mode=refined, warm_start=refined)
        ax = [(np.arange(2 * c, dtype=np.float32) + 0.5) * np.float32(h / 2) for c in cells]
        pos = np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
        vel = np.random.default_rng(sum(cells)).normal(0, 0.5, pos.shape).astype(np.float32)
        pair = []
        for _ in range(2):
            g = bnn.FLIPSolver(params)
            g.set_particles(pos, vel)
            pair.append(g)
        made.append(pair)
    b = Batch()
    for _ in range(2):
        for alone, _ in made:
            alone.step(DT)
        assert np.all(b.step([g for _, g in made], DT) == 0)
    bricks = [alone.stats()["num_active_bricks"] for alone, _ in made]
    assert min(bricks) <= 1024 < max(bricks)
    for alone, g in made:
        assert np.array_equal(alone.pressure(), g.pressure())
        for x, y in zip(alone.particles(), g.particles()):
            assert np.array_equal(x, y)
        for k in ("pcg_iterations", "outer_iterations", "pcg_success", "pcg_residual"):
            assert alone.stats()[k] == g.stats()[k], k
        alone.close()
        g.close()
