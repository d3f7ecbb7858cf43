"""Small maps, whose row segments several waves share (the split form of the direct kernels): every halo type, halo
counts around the number of waves, columns around the 64 of a segment, one row and one pixel, against the
extended oracle with the FP64 criterion of parity.py; FP32C against FP64 within the bounds of
test_gpu_fp32c.py and test_gpu_fp32c_gradient.py; a pixel on a PIEMD centre is NaN in the potential."""
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


def _lens(n, n14=0):
    rng = np.random.default_rng(100 + n)
    halos = []
    for k in range(n - n14):
        halos.append(dict(type=(81, 5, 8)[k % 3], x=float(rng.uniform(-20, 20)), y=float(rng.uniform(-20, 20)),
                          sigma=float(rng.uniform(100, 500)), e=float(rng.uniform(0.02, 0.5)), theta=float(rng.uniform(0, 3.1)),
                          rcore=float(rng.uniform(0.05, 2.0)), rcut=float(rng.uniform(10, 200))))
    halos += [dict(type=14, x=0.0, y=0.0, b0=0.0, epot=0.04, theta=0.3)] * n14
    return M.LensModel.from_halos(halos)


@pytest.mark.parametrize("n,nx,ny", [(1, 1, 1), (7, 65, 3), (8, 64, 5), (9, 63, 2), (23, 130, 7), (66, 200, 11)])
def test_split_maps(hip, oracle, n, nx, ny):
    lens = _lens(n, n14=1 if n > 8 else 0)
    grid = M.Grid(M.grid_param(-21.3, 22.1, -20.7, 21.9), nx, ny, step=(0.213, 0.31))
    print_case("split", lens, grid)
    a, b, c, _ = hip.hessian_grid(lens, grid, 3, 5)
    (ea, eb, ec), (ta, tb, tc) = hessian_reference(oracle, lens, grid, 3, 5)
    for what, got, ex, tol in (("a", a, ea, ta), ("b", b, eb, tb), ("c", c, ec, tc)):
        assert_close(what, got, ex, np.zeros_like(tol), tol)
    for p32, p64 in zip(hip.hessian_grid(lens, grid, 3, 5, precision=hip.PREC_FP32C)[:3], (a, b, c)):
        assert np.abs(p32 - p64).max() <= 2e-7
    lens = lens.subset(np.nonzero(lens.type != 14)[0])
    gx, gy = hip.gradient_grid(lens, grid)
    ex, ey = oracle.gradient_grid(lens, grid, extended=True)
    _, _, sx, sy = oracle.gradient_grid(lens, grid, with_abs=True)
    cg, _ = oracle.cond_planes(lens, grid)
    assert_close("gx", gx, ex, np.zeros_like(sx), REL * sx + EXT_SHARE * cg)
    assert_close("gy", gy, ey, np.zeros_like(sy), REL * sy + EXT_SHARE * cg)
    fx, fy = hip.gradient_grid(lens, grid, precision=hip.PREC_FP32C)
    assert np.hypot(fx - gx, fy - gy).max() <= 2e-5
    # (the gradient's criterion is void on a lone halo's centre, where the sum of the terms is zero)
    at = int(np.nonzero(lens.type != 5)[0][0])
    lens.x[at] = grid.frame.xmin + (nx // 2) * grid.dx
    lens.y[at] = grid.frame.ymin + (ny // 2) * grid.dy
    lens.refresh()
    phi = hip.potential_grid(lens, grid)
    ep = oracle.potential_grid(lens, grid, extended=True)
    S = sum(np.abs(np.nan_to_num(oracle.potential_grid(lens.subset([h]), grid, extended=True))) for h in range(lens.n))
    assert np.isnan(phi[ny // 2, nx // 2])
    np.testing.assert_array_equal(np.isnan(phi), np.isnan(ep))
    fin = ~np.isnan(ep)
    assert_close("phi", np.where(fin, phi, 0.), np.where(fin, ep, 0.), S, np.zeros_like(S))
    m = hip.Model(lens, hip.MAP_POT)
    out = hip.DeviceArray(grid.npix)
    m.map(hip.MAP_POT, 3, [out.ptr], grid, precision=hip.PREC_FP32C)
    hip.sync()
    p32 = out.download().reshape(ny, nx)
    m.close()
    np.testing.assert_array_equal(np.isnan(p32), ~fin)
    assert (np.abs(p32 - phi)[fin] <= 1e-5 * S[fin]).all()


@pytest.mark.parametrize("n,npts", [(1, 1), (7, 64), (8, 65), (23, 63), (66, 129)])
def test_split_points(hip, oracle, n, npts):
    lens = _lens(n)
    rng = np.random.default_rng(npts)
    px, py = rng.uniform(-30, 30, npts), rng.uniform(-30, 30, npts)
    print(f"[case] split points: {n} halos, {npts} points", flush=True)
    gx, gy = hip.point_gradients(lens, px, py)
    for i in range(npts):
        e = oracle.point_gradient(lens, px[i], py[i], extended=True)
        cg, _ = oracle.point_cond(lens, px[i], py[i])
        tol = REL * (np.abs(np.array(e)).max() + 1.0) + EXT_SHARE * cg
        assert abs(gx[i] - e[0]) <= tol and abs(gy[i] - e[1]) <= tol, i
