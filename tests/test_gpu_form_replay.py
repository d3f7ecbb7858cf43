"""The form of maps made beside the replays of a captured sequence that uploads the model's parameters: it follows the
samples on the device, so an eager map after a replay is bit for bit the map of a new model of the lens staged
last, and one before the first replay that of the lens uploaded before."""
import numpy as np
import pytest

from parity import print_case
from test_gpu_form import GRID, _maps, _pair, hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_eager_maps_beside_replays(hip, precision):  # noqa: F811
    lenses = _pair()
    print_case(f"eager fields beside replays, precision={precision}", lenses[0], GRID)
    alone, form = [], []
    for lens in lenses:
        m = hip.Model(lens, hip.MAP_HESSIAN)
        form.append(m.form(hip.MAP_FIELDS, GRID, precision))
        alone.append([p[0] for p in _maps(hip, m, hip.MAP_FIELDS, 5, 1, precision)])
        m.close()
    assert form == ["tiles_64_halves", "pixels"]
    s = hip.stream_create()
    try:
        m = hip.Model(lenses[0], hip.MAP_HESSIAN)
        outs = [hip.DeviceArray(GRID.npix) for _ in range(5)]
        m.stage(lenses[1])
        g = hip.Graph(s)
        m.upload(s)
        m.map(hip.MAP_FIELDS, 1, [o.ptr for o in outs], GRID, r=0.7, precision=precision, stream=s)
        g.end()
        on_device = 0
        for k in (None, 1, 0, 0, 1):
            if k is not None:
                m.stage(lenses[k])
                g.launch()
                hip.sync(s)
                on_device = k
                if k == 1:  # the sequence keeps the form of the lens that was staged at its capture
                    for o, want in zip(outs, alone[1]):
                        np.testing.assert_array_equal(o.download(), want)
            assert m.form(hip.MAP_FIELDS, GRID, precision) == form[on_device]
            for got, want in zip(_maps(hip, m, hip.MAP_FIELDS, 5, 1, precision), alone[on_device]):
                np.testing.assert_array_equal(got[0], want)
        g.close()
        # without the sequence the model goes on as any other
        m.update(lenses[0])
        assert m.form(hip.MAP_FIELDS, GRID, precision) == form[0]
        m.close()
        for o in outs:
            o.close()
    finally:
        hip.stream_destroy(s)


def test_model_freed_before_the_sequence(hip):  # noqa: F811
    """A sequence may outlive a model whose upload it holds, as long as it is not launched any more."""
    lenses = _pair()
    print_case("model destroyed, then the sequence", lenses[0], GRID)
    s = hip.stream_create()
    try:
        m = hip.Model(lenses[0], hip.MAP_HESSIAN)
        g = hip.Graph(s)
        m.upload(s)
        g.end()
        g.launch()
        hip.sync(s)
        m.close()
        g.close()
    finally:
        hip.stream_destroy(s)
