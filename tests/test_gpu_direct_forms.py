"""The direct kernels where the tile expansions and the split form do not take their place (lt_map_form says so): 1, 2
and 4 pixels per thread give the same map bit for bit in every family and precision; the FP32C Hessian,
gradient and potential kernels against the FP64 ones at full size, with the bounds of test_gpu_fp32c.py and
test_gpu_fp32c_gradient.py, on the cluster lens cut into more runs than the expansions take."""
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


def _few(n14):
    rng = np.random.default_rng(6)
    halos = [dict(type=(81, 5, 8)[k % 3], x=float(rng.uniform(-30, 30)), y=float(rng.uniform(-30, 30)),
                  sigma=float(rng.uniform(100, 500)), e=float(rng.uniform(0.02, 0.5)), theta=float(rng.uniform(0, 3.1)),
                  rcore=float(rng.uniform(0.05, 2.0)), rcut=float(rng.uniform(10, 200))) for k in range(6)]
    halos += [dict(type=14, x=0.0, y=0.0, b0=0.0, epot=0.04, theta=0.3)] * n14
    return M.LensModel.from_halos(halos)


def _maps(hip, model, kind, planes, grid, precision, px=0, mode=1):
    outs = [hip.DeviceArray(grid.npix) for _ in range(planes)]
    model.map(kind, mode, [o.ptr for o in outs], grid, r=0.7, precision=precision, px=px)
    hip.sync()
    got = [o.download().reshape(grid.ny, grid.nx) for o in outs]
    for o in outs:
        o.close()
    return got


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("which", ["group", "few"])
def test_px_variants(hip, which, precision):
    grid = M.Grid(M.grid_param(-40, 40, -35, 35), 401, 237)
    modes = [(hip.MAP_FIELDS, 0, 5), (hip.MAP_HESSIAN, 0, 4), (hip.MAP_MASS, 4, 1), (hip.MAP_DPL, 1, 2), (hip.MAP_POT, 1, 1)]
    modes += [(hip.MAP_AMPLI, mode, 1) for mode in range(1, 7)] + [(hip.MAP_SHEAR, mode, 1) for mode in range(1, 5)]
    for kind, mode, planes in modes:
        use = kind if kind in (hip.MAP_MASS, hip.MAP_DPL, hip.MAP_POT) else hip.MAP_HESSIAN
        lens = M.group_lens(seed=4) if which == "group" else _few(0 if kind in (hip.MAP_DPL, hip.MAP_POT) else 1)
        print_case(f"px variants {which} kind {kind} mode {mode} precision={precision}", lens, grid)
        m = hip.Model(lens, use)
        assert m.form(kind, grid, precision) == "pixels"
        first = _maps(hip, m, kind, planes, grid, precision, px=2, mode=mode)
        for px in (1, 4, 0):
            for a, b in zip(_maps(hip, m, kind, planes, grid, precision, px=px, mode=mode), first):
                np.testing.assert_array_equal(a, b)
        m.close()


def _cut_cluster():
    """The 503-halo cluster lens with 17 massless SIS far outside between its halos: 35 runs of the same lens."""
    lens = M.cluster_lens()
    extra = M.LensModel.from_halos([dict(type=5, x=2000.0 + k, y=0.0, b0=0.0, e=0.0) for k in range(17)])
    at = np.linspace(20, lens.n - 20, 17).astype(int)
    fields = ("type", "x", "y", "b0", "angle", "epot", "rcore", "rcut", "z", "dlsds")
    return M.LensModel(*[np.insert(getattr(lens, f), at, getattr(extra, f)) for f in fields])


def test_fp32c_fields_full_size(hip):
    """4096^2: kappa and gamma within 2e-7, det A within 1e-6 of the FP64 kernel; not the same map."""
    lens, grid = _cut_cluster(), M.cluster_grid(4096)
    print_case("FP32C fields, direct", lens, grid)
    m = hip.Model(lens, hip.MAP_HESSIAN)
    maps = []
    for precision in (0, 1):
        assert m.form(hip.MAP_FIELDS, grid, precision) == "pixels"
        maps.append(_maps(hip, m, hip.MAP_FIELDS, 4, grid, precision))
    m.close()
    err = [float(np.abs(a - b).max()) for a, b in zip(*maps)]
    print("max |FP32C - FP64| of kappa, gamma1, gamma2, det A:", err, flush=True)
    assert max(err[:3]) <= 2e-7 and err[3] <= 1e-6 and min(err) > 0


def test_fp32c_gradient_and_potential(hip):
    """1024^2: deflection within 2e-5 arcsec, potential within 1e-5 of the sum of the halos' (a lower bound of it,
    from the 16 largest)."""
    lens, grid = _cut_cluster(), M.cluster_grid(1024)
    print_case("FP32C gradient and potential, direct", lens, grid)
    m = hip.Model(lens, hip.MAP_GRADIENT)
    assert [m.form(hip.MAP_GRADIENT, grid, p) for p in (0, 1)] == ["pixels", "pixels"]
    a, b = (_maps(hip, m, hip.MAP_GRADIENT, 2, grid, p) for p in (0, 1))
    m.close()
    err = float(np.hypot(a[0] - b[0], a[1] - b[1]).max())
    m = hip.Model(lens, hip.MAP_POT)
    assert [m.form(hip.MAP_POT, grid, p) for p in (0, 1)] == ["pixels", "pixels"]
    (a,), (b,) = (_maps(hip, m, hip.MAP_POT, 1, grid, p) for p in (0, 1))
    m.close()
    S = np.zeros_like(a)
    for h in np.argsort(-np.abs(lens.b0))[:16]:
        S += np.abs(hip.potential_grid(lens.subset([h]), grid))
    rel = float((np.abs(a - b) / S).max())
    print(f"max |dalpha| {err:.3e} arcsec, max |dphi| / sum |phi_h| {rel:.3e}", flush=True)
    assert 0 < err <= 2e-5 and 0 < rel <= 1e-5
