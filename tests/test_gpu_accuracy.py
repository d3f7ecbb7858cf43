"""How far maps are from the extended oracle in the 2-norm, by form: the tile expansions and the direct sums of the same
pixels (rows asked for as grids of their own), and point gradients. Bounds: 1e-15 of the norm for the expansions, whose
nodes take fully corrected reciprocals, 2e-15 for the direct sums, whose terms are good to a few units in the last place
(2^-48 reciprocals) and add up over the halos; and the expansions are no farther off than the direct sums."""
import numpy as np
import pytest

import ltmodel as M
from parity import print_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import lthip
    lthip.check(lthip.lib().lt_init(0))
    return lthip


def _norm(got, exact):
    return float(np.sqrt(sum(((g - e) ** 2).sum() for g, e in zip(got, exact)) / sum((e ** 2).sum() for e in exact)))


@pytest.mark.parametrize("halos,n", [(200, 1024), (503, 2048)])
def test_errors(hip, oracle, halos, n):
    lens, grid = M.cluster_lens(seed=1, ngal=halos - 3), M.cluster_grid(n)
    line = M.Grid(grid.frame, n, 1, step=(grid.dx, grid.dy))
    print_case("errors against the extended oracle", lens, grid)
    rows = np.random.default_rng(3).integers(0, n, 8)
    cases = [("Hessian", hip.MAP_HESSIAN, hip.hessian_grid, lambda j: oracle.hessian_planes(lens, line, 0, j, extended=True)[:3]),
             ("gradient", hip.MAP_GRADIENT, hip.gradient_grid, lambda j: oracle.gradient_grid(lens, line, 0, j, extended=True)[:2]),
             ("potential", hip.MAP_POT, hip.potential_grid, lambda j: [oracle.potential_grid(lens, line, 0, j, extended=True)])]
    for name, kind, run, exact in cases:
        m = hip.Model(lens, kind)
        assert m.form(kind, grid).startswith("tiles") and m.form(kind, line) in ("pixels", "parts")
        m.close()
        ex = [exact(int(j)) for j in rows]
        planes = len(ex[0])
        whole = run(lens, grid)
        whole = whole[:planes] if planes > 1 else [whole]
        direct = [run(lens, line, 0, int(j)) for j in rows]
        direct = [d[:planes] if planes > 1 else [d] for d in direct]
        tiles = _norm([w[j] for j in rows for w in whole], [e[0] for x in ex for e in x])
        parts = _norm([d[0] for x in direct for d in x], [e[0] for x in ex for e in x])
        print(f"{name}: {halos} halos, {n}^2: expansions {tiles:.2e}, direct {parts:.2e}", flush=True)
        assert tiles <= 1e-15 and parts <= 2e-15 and tiles <= parts
        if name == "gradient":
            cols = np.random.default_rng(4).integers(0, n, (8, 50))
            px = (grid.frame.xmin + cols * grid.dx).ravel()
            py = (grid.frame.ymin + np.repeat(rows, 50) * grid.dy).ravel()
            got = hip.point_gradients(lens, px, py)
            want = [np.concatenate([e[k][0][c] for e, c in zip(ex, cols)]) for k in (0, 1)]
            points = _norm(got, want)
            print(f"points: {halos} halos: {points:.2e}", flush=True)
            assert points <= 2e-15
