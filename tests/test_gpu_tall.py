"""Maps of one or two columns and more rows than a launch takes work-groups in one dimension when each has a row of
its own: the rows at the ends and around 65535 equal the same rows computed as a small map, within rounding."""
import numpy as np
import pytest

import ltmodel as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1, 65535), (1, 65536), (2, 70001)])
def test_tall_maps(nx, ny):
    import lthip as hip
    hip.check(hip.lib().lt_init(0))
    lens = M.cluster_lens(seed=4, ngal=297)
    grid = M.Grid(M.grid_param(-60., 60., -70., 70.), nx, ny, step=(0.3, 0.002))
    print(f"[case] {nx} columns, {ny} rows", flush=True)
    whole = [*hip.hessian_grid(lens, grid)[:3], *hip.gradient_grid(lens, grid), hip.potential_grid(lens, grid)]
    few = M.Grid(grid.frame, nx, 5, step=(grid.dx, grid.dy))
    for j in (0, 65530, ny - 5):
        part = [*hip.hessian_grid(lens, few, 0, j)[:3], *hip.gradient_grid(lens, few, 0, j), hip.potential_grid(lens, few, 0, j)]
        for w, p in zip(whole, part):
            # sums of 300 terms of one magnitude in another order: a few hundred roundings of the largest value
            assert np.abs(w[j:j + 5] - p).max() <= 300 * 2.2e-16 * np.abs(w).max()
