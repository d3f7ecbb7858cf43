"""Host-array calls whose results pass through the pinned area: planes of less than a piece, of exactly one, just over,
and of several with a remainder, in one thread and in several, equal the device maps bit for bit; point gradients
whose input is larger than the area equal the same points in smaller calls; likelihood calls of changing sizes in turn,
and from two threads, equal their first results (the buffers kept between calls hold nothing of the call before)."""
import threading

import numpy as np
import pytest

import ltmodel as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import lthip
    lthip.check(lthip.lib().lt_init(0))
    return lthip


@pytest.mark.parametrize("nx,ny", [(2, 2), (300, 250), (512, 512), (512, 513), (1031, 1700)])
def test_maps(hip, nx, ny):
    lens = M.group_lens(seed=2)
    grid = M.Grid(M.grid_param(-90., 90., -80., 85.), nx, ny)
    print(f"[case] host planes {nx}x{ny}", flush=True)
    r = hip.cosmo_dlsds(0.4, 2.0, M.flat_lcdm(70.0, 0.3))
    m = hip.Model(lens, hip.MAP_HESSIAN)
    outs = [hip.DeviceArray(grid.npix) for _ in range(5)]
    m.map(hip.MAP_FIELDS, 0, [o.ptr for o in outs], grid, r=r)
    hip.sync()
    for _ in range(2):
        for got, o in zip(hip.map_fields(lens, grid, M.flat_lcdm(70.0, 0.3), 0.4, 2.0), outs):
            np.testing.assert_array_equal(got.ravel(), o.download())
    m.close()


def test_points(hip):
    lens = M.group_lens(seed=2).subset(np.arange(3))
    rng = np.random.default_rng(4)
    n = 1_100_000
    px, py = rng.uniform(-90, 90, n), rng.uniform(-90, 90, n)
    print(f"[case] {n} points", flush=True)
    gx, gy = hip.point_gradients(lens, px, py)
    for a, b in ((0, 1), (1, 131073), (900_000, n)):
        hx, hy = hip.point_gradients(lens, px[a:b], py[a:b])
        np.testing.assert_array_equal(hx, gx[a:b])
        np.testing.assert_array_equal(hy, gy[a:b])


def test_likelihood_calls_in_turn(hip):
    rng = np.random.default_rng(9)
    cases = []
    for n, nsets in ((96, 3), (2500, 9), (64, 70), (300, 1)):  # 2500: more than the kept device buffer
        images = M.galaxies_array(3 * nsets)
        images["cx"], images["cy"] = rng.uniform(-30, 30, (2, 3 * nsets))
        images["dr"] = np.repeat(rng.uniform(0.5, 0.9, nsets), 3)
        cases.append((M.group_lens(seed=n), n, M.grid_param(-80., 80., -80., 80.), np.full(nsets, 3, np.int32), images))
    print("[case] likelihood calls of changing sizes", flush=True)
    first = [hip.chi_barycentersource(*c) for c in cases]
    for c, f in zip(cases, first):
        batch = hip.ChiBatch(1, c[0].type, c[1], c[2], c[3], c[4])
        chi = batch.run([c[0]])[0]
        assert chi[0] == f[1]
    bad = []

    def again(order):
        for k in order:
            if hip.chi_barycentersource(*cases[k]) != first[k]:
                bad.append(k)

    threads = [threading.Thread(target=again, args=(o,)) for o in ((0, 2, 1, 3, 0), (3, 0, 2, 3, 1))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
