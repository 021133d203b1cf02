"""P2G at the edges of its work split: a workgroup owns 14 x 14 node columns and a segment of 2 to 16
planes, so the grids here end just before, on and after those limits, are filled to their last cell,
and hold particles outside the grid (binned to the clamped cell, weights clamped as the reference's).

Bar: valid flags equal the oracle's; face velocities differ by summation order alone. A node's sum has
at most n terms (the particles of its 27 cells); two FP32 orders of n terms, for momentum and for
weight, differ by at most 4 n 2^-24 of the largest node velocity a particle carries.
"""
import numpy as np
import pytest

from banana_amd import scenes
from banana_amd.serving import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [0, 1], ids=["flip", "apic"])
@pytest.mark.parametrize("cells", [(9, 10, 3), (8, 23, 12), (24, 9, 29), (25, 24, 13), (37, 38, 12)])
def test_p2g_tile_edges(oracle, bnn, cells, scheme):
    h = 1.0 / 16.0
    params = scenes.base_params(16)
    params.update(box_max=tuple(c * h for c in cells), transfer_scheme=scheme)
    n, bmin, dx = scenes.grid_dims(params)
    rng = np.random.default_rng(sum(cells) + scheme)
    ext = np.array(n) * np.float64(dx)
    pos = rng.uniform(0, 1, (4 * n[0] * n[1] * n[2], 3)) * ext + bmin
    stray = rng.choice(pos.shape[0], 200, replace=False)
    pos[stray] += rng.choice([-1.0, 1.0], (200, 3)) * rng.uniform(0, 1, (200, 3)) * ext
    pos = pos.astype(np.float32)
    vel = rng.normal(0, 0.5, pos.shape).astype(np.float32)
    aff = rng.normal(0, 2.0, (pos.shape[0], 3, 3)).astype(np.float32)
    g, o = bnn.FLIPSolver(params), oracle.Oracle(params)
    assert g.n == n == o.n
    g.set_particles(pos, vel)
    o.set_particles(pos, vel)
    if scheme:
        g.set_affine(aff)
        o.set_scheme(scheme)
        o.set_affine(aff)
    g.map_particles_to_grid()
    o.map_particles_to_grid()
    _, start = g.bins()
    cnt = np.pad(np.diff(start.astype(np.int64)).reshape(n[2], n[1], n[0]), 1)
    terms = max(int(cnt[k:k + 3, j:j + 3, i:i + 3].sum()) for k in range(n[2]) for j in range(n[1]) for i in range(n[0]))
    carried = np.abs(vel).max()
    if scheme:  # the farthest node a particle reaches: 1.5 cells per axis, or from outside to the clamped node
        far = np.maximum(1.5 * dx, np.maximum(bmin - pos, pos - (bmin + ext)).max(1) + 1.5 * dx)
        carried += (np.abs(aff).max((1, 2)) * 3 * far).max()
    bar = 4 * terms * 2.0 ** -24 * carried
    for c, f, fv in (("u", oracle.F_U, oracle.F_VALID_U), ("v", oracle.F_V, oracle.F_VALID_V), ("w", oracle.F_W, oracle.F_VALID_W)):
        assert np.array_equal(g.grid("valid_" + c), o.field(fv)), c
        assert np.abs(g.grid(c) - o.field(f)).max() <= bar, c
    g.close()


@pytest.mark.parametrize("scheme", [0, 1], ids=["flip", "apic"])
@pytest.mark.parametrize("seg", [4, 8, 16])
def test_p2g_segments(oracle, bnn, seg, scheme):
    """A small grid alone is cut into segments of two planes. The longer ones, through a batch that sets them:
    node planes that end just before, on and after a segment's end (the last segment is then a plane short,
    whole, or one plane), stepped beside the same scenes alone, whose P2G is held to the oracle."""
    h = 1.0 / 16.0
    DT = np.float32(1.0 / 600.0)
    pairs = []
    for k, planes in enumerate((2 * seg - 1, 2 * seg, 2 * seg + 1)):
        cells = (15, 13, planes - 1)
        params = scenes.base_params(16)
        params.update(box_max=tuple(c * h for c in cells), transfer_scheme=scheme, n_expand_cells=0, max_cg_iteration=1)
        n, bmin, dx = scenes.grid_dims(params)
        assert n[2] + 1 == planes
        rng = np.random.default_rng(seg + k)
        pos = (rng.uniform(0, 1, (4 * n[0] * n[1] * n[2], 3)) * np.array(n) * np.float64(dx)).astype(np.float32)
        vel = rng.normal(0, 0.5, pos.shape).astype(np.float32)
        o = oracle.Oracle(params)
        o.set_particles(pos, vel)
        sims = [bnn.FLIPSolver(params) for _ in range(3)]
        for g in sims:
            g.set_particles(pos, vel)
        aff = rng.normal(0, 2.0, (pos.shape[0], 3, 3)).astype(np.float32)
        if scheme:
            o.set_scheme(scheme)
            o.set_affine(aff)
            for g in sims:
                g.set_affine(aff)
        first, alone, batched = sims
        first.map_particles_to_grid()
        o.map_particles_to_grid()
        _, start = first.bins()
        cnt = np.pad(np.diff(start.astype(np.int64)).reshape(n[2], n[1], n[0]), 1)
        terms = max(int(cnt[k:k + 3, j:j + 3, i:i + 3].sum()) for k in range(n[2]) for j in range(n[1]) for i in range(n[0]))
        bar = 4 * terms * 2.0 ** -24 * (np.abs(vel).max() + (np.abs(aff).max() * 3 * 1.5 * dx if scheme else 0))
        for c, f, fv in (("u", oracle.F_U, oracle.F_VALID_U), ("v", oracle.F_V, oracle.F_VALID_V), ("w", oracle.F_W, oracle.F_VALID_W)):
            assert np.array_equal(first.grid("valid_" + c), o.field(fv)), c
            assert np.abs(first.grid(c) - o.field(f)).max() <= bar, c
        first.close()
        pairs.append((alone, batched))
    b = Batch()
    b.set_shape(p2g_segment=seg, graphs=False)
    for _ in range(2):
        for alone, _ in pairs:
            alone.step(DT)
        b.step([g for _, g in pairs], DT)
    assert b.info()["shape"]["p2g_segment"] == seg
    for alone, g in pairs:
        for c in ("u", "v", "w", "old_u", "old_v", "old_w"):  # old: P2G's values, extrapolated and constrained
            assert np.array_equal(alone.grid(c), g.grid(c)), c
        for x, y in zip(alone.particles(), g.particles()):
            assert np.array_equal(x, y)
        alone.close()
        g.close()
