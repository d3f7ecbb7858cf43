"""Batches of small maps. The split form gives a single small map's row segments to eight waves each; a batch fills
the chip with one wave per segment, which forms the same parts one after another: every sample equals its single map
bit for bit (one and two pixels per thread, every halo type, runs of circular SIS, Kmap weights, runs shorter than the parts, both
precisions). And a batch of small maps costs about what the same pixels cost in larger maps."""
import time

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


def _mixed(n, n14=0, circular=False):
    rng = np.random.default_rng(n)
    halos = []
    for k in range(n - n14):
        halos.append(dict(type=(81, 5, 8)[k % 3], x=float(rng.uniform(-50, 50)), y=float(rng.uniform(-50, 50)),
                          sigma=float(rng.uniform(100, 500)), e=float(rng.uniform(0.02, 0.5)) if k % 3 != 1 or not circular else 0.0, theta=float(rng.uniform(0, 3.1)),
                          rcore=float(rng.uniform(0.05, 2.0)), rcut=float(rng.uniform(10, 200))))
    halos += [dict(type=14, x=0.0, y=0.0, b0=0.0, epot=0.04, theta=0.3)] * n14
    return M.LensModel.from_halos(halos)


def _planes(hip, model, kind, mode, grid, nsamples, precision):
    n = {hip.MAP_FIELDS: 5, hip.MAP_HESSIAN: 4, hip.MAP_DPL: 2}.get(kind, 1)
    outs = [hip.DeviceArray(nsamples * grid.npix) for _ in range(n)]
    model.map(kind, mode, [o.ptr for o in outs], grid, r=0.7, precision=precision)
    hip.sync()
    got = [o.download().reshape(nsamples, grid.npix) for o in outs]
    for o in outs:
        o.close()
    return got


@pytest.mark.parametrize("circular", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,nx,ny", [(41, 64, 61), (41, 65, 63), (41, 150, 41), (90, 129, 70), (21, 70, 66)])
def test_batch_equals_single(hip, n, nx, ny, precision, circular):
    grid = M.Grid(M.grid_param(-60, 60, -60, 60), nx, ny)
    print_case(f"batch of small maps precision={precision} circular={circular}", _mixed(n), grid)
    for kind, mode, use, n14, weights in ((hip.MAP_FIELDS, 0, hip.MAP_HESSIAN, 2, False), (hip.MAP_MASS, 4, hip.MAP_MASS, 2, True),
                                          (hip.MAP_HESSIAN, 0, hip.MAP_MASS, 2, True), (hip.MAP_MASS, 4, hip.MAP_MASS, 0, False),
                                          (hip.MAP_DPL, 1, hip.MAP_DPL, 0, False), (hip.MAP_POT, 1, hip.MAP_POT, 0, False)):
        base = _mixed(n, n14, circular)
        if weights:
            base.dlsds[:] = np.where(base.type == 81, 0.7, np.where(base.type == 5, 0.55, 0.62))
            base._soa = None
        samples = M.perturbed_samples(base, 64, seed=3)
        for s in samples:
            s.dlsds[:] = base.dlsds
            s._soa = None
        bm = hip.Model(samples, use)
        got = _planes(hip, bm, kind, mode, grid, len(samples), precision)
        bm.close()
        for k in (0, 31, 63):
            sm = hip.Model(samples[k], use)
            one = _planes(hip, sm, kind, mode, grid, 1, precision)
            sm.close()
            for g, o in zip(got, one):
                np.testing.assert_array_equal(g[k], o[0])


def _time(hip, lens, nsamples, n, precision):
    m = hip.Model(M.perturbed_samples(lens, nsamples, seed=3), hip.MAP_HESSIAN)
    grid = M.Grid(M.grid_param(-60, 60, -60, 60), n, n)
    out = hip.DeviceArray(nsamples * grid.npix)
    best = 1e9
    for _ in range(6):
        t = time.perf_counter()
        for _ in range(20):
            m.map(hip.MAP_AMPLI, 1, [out.ptr], grid, r=0.7, precision=precision)
        hip.sync()
        best = min(best, (time.perf_counter() - t) / 20)
    m.close()
    out.close()
    return best * 1e6


def test_batch_times(hip):
    """Times of the same number of pixels, in us: 256 maps of 100 x 100 of a light lens against 64 of 200 x 200 (1.0
    measured; 2.5 when each row segment went to eight waves), and 256 maps of 100 x 100 of 60 halos in FP32C against
    FP64 (1.3; 3.0)."""
    print("[case] times of batches of small maps", flush=True)
    light = M.group_lens(seed=4)
    for precision in (0, 1):
        small, large = _time(hip, light, 256, 100, precision), _time(hip, light, 64, 200, precision)
        print(f"group lens precision={precision}: 256 x 100^2 {small:.1f} us, 64 x 200^2 {large:.1f} us", flush=True)
        assert small <= 1.8 * large
    f32, f64 = _time(hip, _mixed(60), 256, 100, 1), _time(hip, _mixed(60), 256, 100, 0)
    print(f"60 halos, 256 x 100^2: FP32C {f32:.1f} us, FP64 {f64:.1f} us", flush=True)
    assert f32 <= 2.0 * f64
