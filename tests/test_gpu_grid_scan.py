"""The grid build where its scan and its counting change form: tables of less
than a tile, of no whole number of tiles, around 512 tiles (counted in LDS up
to there) and above 1,024 (several scan workgroups); particles in long runs of
one cell, in random order and around a wave's count; each grid built twice."""
import numpy as np
import pytest

from psb_project_amd import scenes
from psb_project_amd._lib import check, lib
from tests.test_gpu_parity import _grid, _grid_arrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["runs", "random"])
@pytest.mark.parametrize("dims,n", [((3, 3, 3), 1), ((16, 16, 16), 64), ((17, 13, 29), 65),
                                    ((128, 128, 128), 5000), ((128, 128, 129), 5000),
                                    ((161, 163, 169), 3001), ((200, 190, 240), 20011)])
def test_grid_tables(ctx, oracle, dims, n, order):
    gd = scenes.wcsph_dam_break(n_side=4).params.grid
    for k in range(3):
        gd.dims[k] = dims[k]
    rng = np.random.default_rng(n)
    lo, cell = np.array(list(gd.min)), gd.cell_size
    ncells = dims[0] * dims[1] * dims[2]
    g = _grid(ctx, gd, n)
    try:
        for turn in range(2):
            x = np.zeros((n, 4), np.float32)
            c = rng.integers(0, np.array(dims), size=(n, 3))
            if order == "runs":   # few cells, many particles in each, one after another
                c = np.repeat(c[: n // 40 + 1], 40, axis=0)[:n]
            x[:, :3] = lo + (c + rng.uniform(0.05, 0.95, (n, 3))) * cell
            check(lib().psb_store_particles(g, ctx.to_device(x).ptr, n))
            hash_, perm, start = _grid_arrays(ctx, g, n, ncells)
            h, p, s, _ = oracle.grid_build(x, gd)
            order_ = np.argsort(h, kind="stable")
            assert np.array_equal(start, s)
            assert np.array_equal(perm, p) and np.array_equal(perm, order_)
            assert np.array_equal(hash_, h)
    finally:
        lib().psb_finalize_grid(g)
