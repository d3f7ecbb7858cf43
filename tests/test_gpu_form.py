"""The form of a halo sum (lt_map_form) follows the sample: two lenses of one model, spread over the map or crowded at
its middle, take different forms, and each gives the same map bit for bit alone, in a batch at any place, after
updates in either order, and as a model of its own; a captured sequence keeps the form of its capture."""
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


def _mixed(n):
    rng = np.random.default_rng(5)
    halos = [dict(type=81, x=0.0, y=0.0, sigma=950.0, e=0.3, theta=0.4, rcore=9.0, rcut=900.0)]
    for k in range(n - 1):
        f = 10.0 ** (0.4 * (18 - rng.uniform(18, 24)))
        halos.append(dict(type=(5, 8, 81)[k % 3], x=float(rng.uniform(-110, 110)), y=float(rng.uniform(-110, 110)),
                          sigma=180.0 * f ** 0.25, e=float(rng.uniform(0.02, 0.6)), theta=float(rng.uniform(0, 3.1)),
                          rcore=0.15 * f ** 0.5, rcut=40.0 * f ** 0.5))
    return M.LensModel.from_halos(halos)


def _pair():
    """(spread, crowded): the same halos over 220 and over 18 arcseconds."""
    spread = _mixed(160)
    crowded = spread.subset(np.arange(spread.n))
    crowded.x *= 0.08
    crowded.y *= 0.08
    crowded.refresh()
    return spread, crowded


GRID = M.Grid(M.grid_param(-110, 110, -110, 110), 673, 577)
# (kind, use, planes, precisions, the crowded lens's form): FP32C mass and potential maps of this size stay direct for both
KINDS = [("MAP_FIELDS", "MAP_HESSIAN", 5, (0, 1), "pixels"), ("MAP_DPL", "MAP_DPL", 2, (0, 1), "parts"),
         ("MAP_MASS", "MAP_MASS", 1, (0,), "pixels"), ("MAP_POT", "MAP_POT", 1, (0,), "parts")]


def _maps(hip, model, kind, planes, nsamples, precision):
    outs = [hip.DeviceArray(nsamples * GRID.npix) for _ in range(planes)]
    model.map(kind, 1, [o.ptr for o in outs], GRID, r=0.7, precision=precision)
    hip.sync()
    got = [o.download().reshape(nsamples, GRID.npix) for o in outs]
    for o in outs:
        o.close()
    return got


@pytest.mark.parametrize("name,use,planes,precisions,direct", KINDS)
def test_form_follows_the_sample(hip, name, use, planes, precisions, direct):
    kind, use = getattr(hip, name), getattr(hip, use)
    lenses, forms = _pair(), ("tiles_64_halves", direct)
    for precision in precisions:
        print_case(f"{name} spread and crowded, precision={precision}", lenses[0], GRID)
        alone = []
        for lens, form in zip(lenses, forms):
            m = hip.Model(lens, use)
            assert m.form(kind, GRID, precision) == form
            alone.append(_maps(hip, m, kind, planes, 1, precision))
            m.close()
        for first in (0, 1):  # a batch whose first sample takes one form or the other, then updated to the other order
            order = [first, 1 - first, 1 - first, first]
            m = hip.Model([lenses[k] for k in order], use)
            for turn in range(2):
                assert [m.form(kind, GRID, precision, sample=s) for s in range(4)] == [forms[k] for k in order]
                got = _maps(hip, m, kind, planes, 4, precision)
                for p in range(planes):
                    for s, k in enumerate(order):
                        np.testing.assert_array_equal(got[p][s], alone[k][p][0])
                order = order[1:] + order[:1]
                m.update_batch([lenses[k] for k in order])
            m.close()
        m = hip.Model(lenses[0], use)
        for k in (1, 0, 1):
            m.update(lenses[k])
            for got, want in zip(_maps(hip, m, kind, planes, 1, precision), alone[k]):
                np.testing.assert_array_equal(got, want)
        m.close()


def test_stage_alone_changes_nothing(hip):
    """lt_model_stage is host work: until the upload, maps and their form are those of the samples on the device."""
    spread, crowded = _pair()
    print_case("stage without upload", spread, GRID)
    m = hip.Model(spread, hip.MAP_HESSIAN)
    want = _maps(hip, m, hip.MAP_FIELDS, 5, 1, 0)
    m.stage(crowded)
    assert m.form(hip.MAP_FIELDS, GRID) == "tiles_64_halves"
    for a, b in zip(_maps(hip, m, hip.MAP_FIELDS, 5, 1, 0), want):
        np.testing.assert_array_equal(a, b)
    m.upload()
    assert m.form(hip.MAP_FIELDS, GRID) == "pixels"
    m.close()


def test_capture_keeps_its_form(hip):
    """Replays of a sequence captured with one lens, staged with the other and back: the captured lens bit for bit,
    the other within rounding (1e-12 of the Hessian's scale at each pixel)."""
    lenses = _pair()
    print_case("captured upload and Hessian", lenses[0], GRID)
    alone = []
    for lens in lenses:
        m = hip.Model(lens, hip.MAP_HESSIAN)
        alone.append([p[0] for p in _maps(hip, m, hip.MAP_HESSIAN, 4, 1, 0)])
        m.close()
    s = hip.stream_create()
    try:
        m = hip.Model(lenses[0], hip.MAP_HESSIAN)
        outs = [hip.DeviceArray(GRID.npix) for _ in range(4)]
        g = hip.Graph(s)
        m.upload(s)
        m.map(hip.MAP_HESSIAN, 0, [o.ptr for o in outs], GRID, stream=s)
        g.end()
        for k in (0, 1, 0, 1):
            m.stage(lenses[k])
            g.launch()
            hip.sync(s)
            scale = sum(np.abs(p) for p in alone[k]) + 1.0
            for o, want in zip(outs, alone[k]):
                got = o.download()
                if k == 0:
                    np.testing.assert_array_equal(got, want)
                else:
                    assert (np.abs(got - want) <= 1e-12 * scale).all()
            other = hip.Model(lenses[1 - k], hip.MAP_HESSIAN)  # eager work between the replays
            _maps(hip, other, hip.MAP_HESSIAN, 4, 1, 0)
            other.close()
        g.close()
        m.close()
    finally:
        hip.stream_destroy(s)


@pytest.mark.parametrize("precision", [0, 1])
def test_kappa_is_half_the_trace(hip, precision):
    """Amplification mode 5 (kappa) is (a + c) / 2 of the Hessian map bit for bit, expanded or direct. (Not so where the
    FP32C kernel runs: its amplification maps take pixels of large kappa again in FP64, its Hessian maps do not.)"""
    for lens, form in zip(_pair()[:2 - precision], ("tiles_64_halves", "pixels")):
        print_case(f"kappa {form} precision={precision}", lens, GRID)
        m = hip.Model(lens, hip.MAP_HESSIAN)
        assert m.form(hip.MAP_AMPLI, GRID, precision) == m.form(hip.MAP_HESSIAN, GRID, precision) == form
        a, _, c, _ = _maps(hip, m, hip.MAP_HESSIAN, 4, 1, precision)
        out = hip.DeviceArray(GRID.npix)
        m.map(hip.MAP_AMPLI, 5, [out.ptr], GRID, r=0.7, precision=precision)
        hip.sync()
        np.testing.assert_array_equal(out.download(), 0.5 * (a[0] + c[0]))
        m.close()


@pytest.mark.parametrize("power", [70, -70])
def test_units(hip, power):
    """A lens and its grid in units of 2^-70 and 2^70 arcseconds: the same Hessian (whose halo terms scale exactly),
    within the rounding between forms (1e-12 of its scale). Maps this far from 1 stay direct: the far tests of the
    expansions square lengths in FP32."""
    lens = _pair()[0]
    print_case(f"units of 2^{-power} arcseconds", lens, GRID)
    m = hip.Model(lens, hip.MAP_HESSIAN)
    want = [p[0] for p in _maps(hip, m, hip.MAP_HESSIAN, 4, 1, 0)]
    m.close()
    unit = 2.0 ** power
    scaled = lens.subset(np.arange(lens.n))
    for f in ("x", "y", "b0", "rcore", "rcut"):
        getattr(scaled, f)[:] *= unit
    scaled.refresh()
    grid = M.Grid(M.grid_param(-110 * unit, 110 * unit, -110 * unit, 110 * unit), GRID.nx, GRID.ny)
    m = hip.Model(scaled, hip.MAP_HESSIAN)
    outs = [hip.DeviceArray(grid.npix) for _ in range(4)]
    m.map(hip.MAP_HESSIAN, 0, [o.ptr for o in outs], grid)
    hip.sync()
    assert m.form(hip.MAP_HESSIAN, grid) == "pixels"
    m.close()
    scale = sum(np.abs(p) for p in want) + 1.0
    for o, w in zip(outs, want):
        assert (np.abs(o.download() - w) <= 1e-12 * scale).all()


@pytest.mark.parametrize("norm", [2.5, 0.4])
def test_angles_of_another_norm(hip, norm):
    """cos and sin of the angles are the caller's: of norm 2.5 and 0.4 a halo's frame is larger or smaller than the lab's
    by that factor. The expanded Hessian at 100 x 60 pixels equals the direct one of that part of the map (1e-12)."""
    lens = _pair()[0]
    lens.cos *= norm
    lens.sin *= norm
    lens._soa = None
    print_case(f"angles of norm {norm}", lens, GRID)
    m = hip.Model(lens, hip.MAP_HESSIAN)
    assert m.form(hip.MAP_HESSIAN, GRID).startswith("tiles")
    whole = [p[0].reshape(GRID.ny, GRID.nx) for p in _maps(hip, m, hip.MAP_HESSIAN, 4, 1, 0)]
    part = M.Grid(GRID.frame, 100, 60, step=(GRID.dx, GRID.dy))
    worst = 0.0
    for i0, j0 in ((0, 0), (290, 260), (573, 517), (100, 400)):
        assert m.form(hip.MAP_HESSIAN, part, istart=i0, jstart=j0) in ("pixels", "parts")
        outs = [hip.DeviceArray(part.npix) for _ in range(4)]
        m.map(hip.MAP_HESSIAN, 0, [o.ptr for o in outs], part, istart=i0, jstart=j0)
        hip.sync()
        got = [o.download().reshape(part.ny, part.nx) for o in outs]
        scale = sum(np.abs(g) for g in got) + 1.0
        for g, w in zip(got, whole):
            worst = max(worst, float((np.abs(w[j0:j0 + 60, i0:i0 + 100] - g) / scale).max()))
    m.close()
    print(f"norm {norm}: {worst:.2e}", flush=True)
    assert worst <= 1e-12


def test_autotune(hip):
    """A map in tiles or in parts has no pixels per thread to tune: one time, given three times, and the default stays
    what a direct map of the same octaves of halos and pixels had it tuned to."""
    spread, crowded = _pair()
    small = M.Grid(GRID.frame, 97, 83)
    print_case("autotune", spread, GRID)
    m = hip.Model(crowded, hip.MAP_HESSIAN)
    assert m.form(hip.MAP_FIELDS, GRID) == "pixels"
    px, ms = m.autotune(hip.MAP_FIELDS, 0, GRID)
    assert px in (1, 2, 4) and len(set(ms)) > 1
    m.close()
    m = hip.Model(spread, hip.MAP_HESSIAN)
    for grid, form in ((GRID, "tiles_64_halves"), (small, "parts")):
        assert m.form(hip.MAP_FIELDS, grid) == form
        best, ms = m.autotune(hip.MAP_FIELDS, 0, grid)
        assert ms[0] == ms[1] == ms[2] > 0
        assert best == (px if grid is GRID else 2)
    m.close()
