"""Active-brick tables on grids of more bricks than one pass of the index holds, with rows that end inside a
4-cell load: fluid cells and active bricks equal those of the level set, and the pressure's order follows."""
import numpy as np
import pytest

from banana_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(170, 171, 172), (401, 150, 45), (5, 6, 7)])
def test_active_bricks_match_level_set(bnn, cells):
    h = 1.0 / 64.0
    params = scenes.base_params(64)
    params.update(box_max=tuple(c * h for c in cells))
    rng = np.random.default_rng(3)
    pos = rng.uniform(0, 1, (3000, 3)) * np.array(cells) * h  # scattered drops: a few cells in most bricks
    pos = np.concatenate([pos, rng.uniform(0, 3 * h, (200, 3))]).astype(np.float32)
    g = bnn.FLIPSolver(params)
    g.set_particles(pos, rng.normal(0, 0.2, pos.shape).astype(np.float32))
    g.step(np.float32(1e-6))
    fluid = g.grid("phi") < 0
    nz, ny, nx = fluid.shape
    pad = np.zeros(tuple(-(-s // 8) * 8 for s in fluid.shape), bool)
    pad[:nz, :ny, :nx] = fluid
    bricks = pad.reshape(pad.shape[0] // 8, 8, pad.shape[1] // 8, 8, pad.shape[2] // 8, 8).any((1, 3, 5))
    st = g.stats()
    assert st["pcg_success"] == 1
    assert st["num_active_cells"] == fluid.sum() and st["num_active_bricks"] == bricks.sum()
    assert g.pressure().shape[0] == fluid.sum()
    g.close()
