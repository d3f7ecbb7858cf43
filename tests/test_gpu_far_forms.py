"""The tile expansions' forms, each shown to run (lt_map_form) where it is held to the extended oracle: Hessian (Kmap
weights too), its trace, gradient and potential on ragged grids with an offset that cuts the first tiles, rows on
and next to the edges of tiles, quarters and the grid, with the criteria of test_gpu_far.py; the cases of
test_gpu_far.py and test_gpu_far_parts.py by the forms that they reach; batches on pitched planes in the forms of
4 and of 16 waves."""
import numpy as np
import pytest

import ltmodel as M
import test_gpu_far as far
import test_gpu_far_parts as parts
from parity import assert_close, hessian_reference, print_case
from test_gpu_far import hip  # noqa: F401

pytestmark = pytest.mark.gpu

GRIDS = {
    "tiles_64": lambda: (far._mixed(64, n14=1), far._grid(110.0, 1473, 1409), 5, 17),
    "tiles_64_wide": lambda: (far._mixed(258, n14=2), far._grid(40.0, 1857, 929), 5, 17),
    "tiles_64_halves": parts.PARTS["halves_cut"],
    "tiles_64_quarters": parts.PARTS["quarters_cut"],
    "tiles_128": far.CASES["root128"],
    "tiles_256": far.CASES["root256"],
}
# the form of each kind's map where it is not the one that names the grid
OTHER = {("tiles_64_quarters", "MAP_MASS"): "pixels", ("tiles_128", "MAP_MASS"): "tiles_64_halves"}


def _model(hip, lens, kind):  # noqa: F811
    use = hip.MAP_HESSIAN if kind in (hip.MAP_HESSIAN, hip.MAP_FIELDS, hip.MAP_AMPLI, hip.MAP_SHEAR) else kind
    if kind in (hip.MAP_GRADIENT, hip.MAP_DPL, hip.MAP_POT):
        lens = lens.subset(np.nonzero(lens.type != 14)[0])
    return hip.Model(lens, use)


@pytest.mark.parametrize("name", GRIDS)
def test_forms(hip, oracle, monkeypatch, name):  # noqa: F811
    lens, grid, i0, j0 = GRIDS[name]()
    for kind in ("MAP_HESSIAN", "MAP_FIELDS", "MAP_AMPLI", "MAP_MASS", "MAP_GRADIENT", "MAP_DPL", "MAP_POT"):
        m = _model(hip, lens, getattr(hip, kind))
        assert m.form(getattr(hip, kind), grid, istart=i0, jstart=j0) == OTHER.get((name, kind), name), kind
        m.close()
    if name in ("tiles_64", "tiles_64_wide"):  # the others' Hessian, gradient and potential: the two modules above
        monkeypatch.setitem(far.CASES, name, GRIDS[name])
        for kmap in (False, True):
            far.test_hessian(hip, oracle, name, kmap)
        far.test_gradient_and_potential(hip, oracle, name)
    # the trace: a mass map is (a + c) / 2 of the weighted Hessian
    lens.dlsds[:] = np.where(lens.type == 81, 0.7, np.where(lens.type == 5, 0.55, 0.62))
    lens._soa = None
    print_case(f"far trace {name}", lens, grid)
    m = hip.Model(lens, hip.MAP_MASS)
    out = hip.DeviceArray(grid.npix)
    m.map(hip.MAP_MASS, 1, [out.ptr], grid, istart=i0, jstart=j0)
    hip.sync()
    kappa = out.download().reshape(grid.ny, grid.nx)
    m.close()
    line = M.Grid(grid.frame, grid.nx, 1, step=(grid.dx, grid.dy))
    for j in far._rows(grid):
        (ea, _, ec), (ta, _, tc) = hessian_reference(oracle, lens, line, i0, j0 + j, kmap=True)
        assert_close(f"kappa row {j}", kappa[j:j + 1], (ea + ec) / 2, np.zeros_like(ta), (ta + tc) / 2)


@pytest.mark.parametrize("module,name,form", [
    ("far", "root64", "pixels"), ("far", "wide", "tiles_64_halves"), ("far", "wide_64halos", "tiles_64_halves"),
    ("parts", "quarters", "tiles_64_quarters"), ("parts", "halves", "tiles_64_halves")])
def test_forms_of_the_other_modules(hip, module, name, form):  # noqa: F811
    lens, grid, i0, j0 = (far.CASES if module == "far" else parts.PARTS)[name]()
    for kind in (hip.MAP_HESSIAN, hip.MAP_GRADIENT, hip.MAP_POT):
        m = _model(hip, lens, kind)
        assert m.form(kind, grid, istart=i0, jstart=j0) == form
        m.close()


@pytest.mark.parametrize("name,pitch", [("tiles_64", 1536), ("tiles_64_quarters", 512)])
def test_batch_and_pitch(hip, name, pitch):  # noqa: F811
    """Two samples in one launch on pitched planes: each equals its single map, and the padding stays."""
    lens, grid, i0, j0 = GRIDS[name]()
    for kind, mode, planes in ((hip.MAP_AMPLI, 3, 1), (hip.MAP_SHEAR, 1, 1), (hip.MAP_DPL, 1, 2), (hip.MAP_POT, 1, 1)):
        samples = M.perturbed_samples(lens if kind in (hip.MAP_AMPLI, hip.MAP_SHEAR) else lens.subset(np.nonzero(lens.type != 14)[0]), 2, seed=4)
        use = hip.MAP_HESSIAN if kind in (hip.MAP_AMPLI, hip.MAP_SHEAR) else kind
        print_case(f"far batch {name} kind {kind}", samples[0], grid)
        bm = hip.Model(samples, use)
        assert [bm.form(kind, grid, sample=s, istart=i0, jstart=j0) for s in (0, 1)] == [name, name]
        outs = [hip.DeviceArray(2 * grid.ny * pitch) for _ in range(planes)]
        for o in outs:
            o.upload(np.full(o.n, 7.0))
        bm.map(kind, mode, [o.ptr for o in outs], grid, r=0.7, pitch=pitch, istart=i0, jstart=j0)
        hip.sync()
        got = [o.download().reshape(2, grid.ny, pitch) for o in outs]
        bm.close()
        for s, one_lens in enumerate(samples):
            sm = hip.Model(one_lens, use)
            one = [hip.DeviceArray(grid.npix) for _ in range(planes)]
            sm.map(kind, mode, [o.ptr for o in one], grid, r=0.7, istart=i0, jstart=j0)
            hip.sync()
            for g, o in zip(got, one):
                np.testing.assert_array_equal(g[s, :, :grid.nx], o.download().reshape(grid.ny, grid.nx))
                assert (g[s, :, grid.nx:] == 7.0).all()
            sm.close()
