"""Maps by tile expansions (lt_far.hip), in each of its work-group shapes, against the extended oracle with
the FP64 criterion of parity.py, at rows on and next to the edges of tiles, quarters and the grid: ragged grids, a
grid offset that cuts the first tile, every halo type (external shear and Kmap weights with the Hessian),
models that end inside and on a 64-halo mask word, a pixel on a PIEMD centre. The tolerance is the direct
kernels' own (1e-12 of the sum of the terms' magnitudes). Then: a part of a map equals the same pixels
of the whole, and a batch its single maps, bit for bit."""
import numpy as np
import pytest

import ltmodel as M
from parity import EXT_SHARE, REL, assert_close, hessian_reference, print_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import lthip
    lthip.check(lthip.lib().lt_init(0))
    return lthip


def _mixed(n, n14=0, seed=5):
    rng = np.random.default_rng(seed)
    halos = [dict(type=81, x=0.0, y=0.0, sigma=950.0, e=0.3, theta=0.4, rcore=9.0, rcut=900.0)]
    for k in range(n - 1 - n14):
        f = 10.0 ** (0.4 * (18 - rng.uniform(18, 24)))
        halos.append(dict(type=(5, 8, 81)[k % 3], x=float(rng.uniform(-110, 110)), y=float(rng.uniform(-110, 110)),
                          sigma=180.0 * f ** 0.25, e=float(rng.uniform(0.02, 0.6)), theta=float(rng.uniform(0, 3.1)),
                          rcore=0.15 * f ** 0.5, rcut=40.0 * f ** 0.5))
    halos += [dict(type=14, x=0.0, y=0.0, b0=0.0, epot=0.04, theta=0.3 + k) for k in range(n14)]
    return M.LensModel.from_halos(halos)


def _grid(half, nx, ny):
    return M.Grid(M.grid_param(-half, half, -half, half), nx, ny)


# (shape, lens, grid, istart, jstart): 4 waves and 16 waves per 64 pixels, roots of 128 and 256 pixels
CASES = {
    "root64": lambda: (M.group_lens(seed=3), _grid(40.0, 961, 897), 0, 0),
    "wide": lambda: (_mixed(160, n14=2), _grid(110.0, 701, 643), 5, 17),
    "wide_64halos": lambda: (_mixed(64), _grid(110.0, 897, 705), 0, 0),
    "root128": lambda: (M.cluster_lens(seed=8, ngal=497), M.Grid(M.grid_param(-150, 150, -150, 150), 517, 389, step=(0.07, 0.08)),
                        1500, 1801),
    "root256": lambda: (M.cluster_lens(seed=9, ngal=1997), M.Grid(M.grid_param(-150, 150, -150, 150), 530, 300, step=(0.03, 0.03)),
                        5000, 4999),
}
ROWS = (0, 1, 31, 32, 63, 64, 127, 128, 255, 256)


def _rows(grid):
    return sorted({r for r in ROWS if r < grid.ny} | {grid.ny - 2, grid.ny - 1})


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("kmap", [False, True])
def test_hessian(hip, oracle, name, kmap):
    lens, grid, i0, j0 = CASES[name]()
    if kmap:
        lens.dlsds[:] = np.where(lens.type == 81, 0.7, np.where(lens.type == 5, 0.55, 0.62))
        lens._soa = None
    print_case(f"far hessian {name} kmap={kmap}", lens, grid)
    a, b, c, d = hip.hessian_grid(lens, grid, i0, j0, kmap=kmap)
    np.testing.assert_array_equal(b, d)
    line = M.Grid(grid.frame, grid.nx, 1, step=(grid.dx, grid.dy))
    for j in _rows(grid):
        (ea, eb, ec), (ta, tb, tc) = hessian_reference(oracle, lens, line, i0, j0 + j, kmap=kmap)
        for what, got, ex, tol in (("a", a, ea, ta), ("b", b, eb, tb), ("c", c, ec, tc)):
            assert_close(f"{what} row {j}", got[j:j + 1], ex, np.zeros_like(tol), tol)
    if name in ("root128", "root256"):
        sub = M.Grid(grid.frame, 150, 90, step=(grid.dx, grid.dy))
        for got, whole in zip(hip.hessian_grid(lens, sub, i0 + 61, j0 + 35, kmap=kmap), (a, b, c, d)):
            np.testing.assert_array_equal(got, whole[35:125, 61:211])


@pytest.mark.parametrize("name", CASES)
def test_gradient_and_potential(hip, oracle, name):
    lens, grid, i0, j0 = CASES[name]()
    lens = lens.subset(np.nonzero(lens.type != 14)[0])
    at = int(np.nonzero(lens.type != 5)[0][0])  # a PIEMD or dPIE halo moves onto a pixel
    lens.x[at] = grid.frame.xmin + (i0 + 33) * grid.dx
    lens.y[at] = grid.frame.ymin + (j0 + 31) * grid.dy
    lens.refresh()
    print_case(f"far gradient, potential {name}", lens, grid)
    gx, gy = hip.gradient_grid(lens, grid, i0, j0)
    phi = hip.potential_grid(lens, grid, i0, j0)
    xs = grid.frame.xmin + (i0 + np.arange(grid.nx)) * grid.dx
    ys = grid.frame.ymin + (j0 + np.arange(grid.ny)) * grid.dy
    centres = np.zeros(phi.shape, bool)  # the pixels on a PIEMD centre: the one placed above, perhaps others
    for h in np.nonzero(lens.type != 5)[0]:
        centres |= (ys == lens.y[h])[:, None] & (xs == lens.x[h])[None, :]
    assert centres[31, 33]
    np.testing.assert_array_equal(np.isnan(phi), centres)
    line = M.Grid(grid.frame, grid.nx, 1, step=(grid.dx, grid.dy))
    for j in _rows(grid)[::2 if lens.n > 500 else 1]:
        ex, ey = oracle.gradient_grid(lens, line, i0, j0 + j, extended=True)
        _, _, sx, sy = oracle.gradient_grid(lens, line, i0, j0 + j, with_abs=True)
        cg, _ = oracle.cond_planes(lens, line, i0, j0 + j)
        assert_close(f"gx row {j}", gx[j:j + 1], ex, np.zeros_like(sx), REL * sx + EXT_SHARE * cg)
        assert_close(f"gy row {j}", gy[j:j + 1], ey, np.zeros_like(sy), REL * sy + EXT_SHARE * cg)
        ep = oracle.potential_grid(lens, line, i0, j0 + j, extended=True)
        fin = np.isfinite(ep)
        assert (np.isfinite(phi[j:j + 1]) == fin).all()
        # the sum of |phi_h| from the 16 largest halos: a lower bound, so a tighter tolerance
        S = np.zeros_like(ep)
        for h in np.argsort(-np.abs(lens.b0))[:16]:
            S += np.abs(np.nan_to_num(oracle.potential_grid(lens.subset([h]), line, i0, j0 + j, extended=True)))
        assert_close(f"phi row {j}", np.where(fin, phi[j:j + 1], 0.), np.where(fin, ep, 0.), S, np.zeros_like(S))


def test_batch_and_pitch(hip):
    """Two samples in one launch on pitched planes: each equals its single map, and the padding stays."""
    samples = M.perturbed_samples(M.group_lens(seed=3), 2, seed=4)
    grid, pitch = _grid(40.0, 961, 897), 1024
    print_case("far batch", samples[0], grid)
    for kind, mode, planes in ((hip.MAP_AMPLI, 3, 1), (hip.MAP_MASS, 4, 1), (hip.MAP_AMPLI, 5, 1), (hip.MAP_DPL, 1, 2)):
        use = {hip.MAP_MASS: hip.MAP_MASS, hip.MAP_DPL: hip.MAP_DPL}.get(kind, hip.MAP_HESSIAN)
        bm = hip.Model(samples, use)
        outs = [hip.DeviceArray(2 * grid.ny * pitch) for _ in range(planes)]
        for o in outs:
            o.upload(np.full(o.n, 7.0))
        bm.map(kind, mode, [o.ptr for o in outs], grid, r=0.7, pitch=pitch)
        hip.sync()
        got = [o.download().reshape(2, grid.ny, pitch) for o in outs]
        bm.close()
        for s, lens in enumerate(samples):
            sm = hip.Model(lens, use)
            one = [hip.DeviceArray(grid.npix) for _ in range(planes)]
            sm.map(kind, mode, [o.ptr for o in one], grid, r=0.7)
            hip.sync()
            for g, o in zip(got, one):
                np.testing.assert_array_equal(g[s, :, :grid.nx], o.download().reshape(grid.ny, grid.nx))
                assert (g[s, :, grid.nx:] == 7.0).all()
            sm.close()
