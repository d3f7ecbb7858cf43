"""Amplification in magnitudes (mode 3, -2.5 log10 |det A|) against 80-bit logarithms, through the epilogue on planes
whose det A is known exactly (a = c, b = 0: det A = fl((1 - a)^2)): over the whole range of doubles, near |det A| = 1
and through it. The error is at most 0.75 units in the last place (0.52 expected: one rounding at the result's size;
1.2 with the library's log10, 3.0 with a logarithm good to 3)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import lthip
    lthip.check(lthip.lib().lt_init(0))
    return lthip


def _magnitudes(hip, a):
    n = len(a)
    da, db, out = hip.DeviceArray(n), hip.DeviceArray(n), hip.DeviceArray(n)
    da.upload(a)
    db.upload(np.zeros(n))
    hip.check(hip.lib().lt_map_epilogue_device(hip.MAP_AMPLI, 3, C.c_void_p(out.ptr), None, None, None, None,
                                               C.c_void_p(da.ptr), C.c_void_p(db.ptr), C.c_void_p(da.ptr), n, 1.0, 1.0, None))
    hip.sync()
    v = out.download()
    for d in (da, db, out):
        d.close()
    return v


@pytest.mark.parametrize("which", ["range", "near", "through"])
def test_magnitudes(hip, which):
    rng = np.random.default_rng(7)
    n = 400000
    if which == "range":  # sqrt |det A| from 2^-53 (as 1 - a has it) and from 2^499 down
        k = rng.uniform(-52, 499, n)
        a = 1.0 - np.exp2(k)
    elif which == "near":
        a = rng.uniform(-0.4, 0.4, n)
    else:
        a = rng.uniform(-1.0, 1.0, n) * np.exp2(rng.uniform(-52, -3, n))
    print(f"[case] magnitudes {which}, {n} values", flush=True)
    det = (1.0 - a) ** 2
    keep = det > 0
    got = _magnitudes(hip, a)[keep]
    exact = np.longdouble(-2.5) * np.log10(det[keep].astype(np.longdouble))
    zero = det[keep] == 1.0
    assert (got[zero] == 0.0).all()
    ulp = np.spacing(np.abs(exact[~zero].astype(np.float64)))
    err = np.abs((got[~zero].astype(np.longdouble) - exact[~zero]) / ulp).astype(np.float64)
    print(f"magnitudes {which}: worst {err.max():.3f} ulp, rms {np.sqrt((err ** 2).mean()):.3f}", flush=True)
    assert err.max() <= 0.75


def test_limits(hip):
    """det A of 0, infinity and NaN."""
    print("[case] magnitudes at the limits", flush=True)
    v = _magnitudes(hip, np.array([1.0, np.inf, np.nan, 1e200, 0.0]))
    assert v[0] == np.inf and np.isnan(v[2]) and v[3] == -np.inf and v[4] == 0.0 and not np.isfinite(v[1])
