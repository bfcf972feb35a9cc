"""Mean flux profiles of a state with one value that is not finite: the same
infinities and NaN as the formula's (3dmhdsub.f:1650-1661), the mean of the
plane's T before the flux about it; finite on the other planes."""

import numpy as np
import pytest

import helpers as H
from test_gpu_stage_split import _box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 0.0])
@pytest.mark.parametrize("field", ["rw", "ru", "ro", "tt"])
def test_profiles_of_one_bad_value(field, value):
    meta, st = _box(16, 9, 5, False)
    st[field][4, 6, 3] = value
    st["tt"][1:-1, 1:-1, 4] = 1.25  # (the flux about a constant T has no correction)
    st["rw"][7, 3, 4] = value
    with H.pkg().Box(meta) as box:
        box.upload(st)
        got = box.flux_profiles()
    ru, rv, rw, ro, tt = (st[k][1:-1, 1:-1, 1:-1] for k in ("ru", "rv", "rw", "ro", "tt"))
    with np.errstate(all="ignore"):
        ri, ttm = 1.0 / ro, tt.mean((0, 1))
        u2 = (ru * ri) ** 2 + (rv * ri) ** 2 + (rw * ri) ** 2
        want = dict(ttm=ttm, rom=ro.mean((0, 1)), fconm=(-(rw * (2.5 * (tt - ttm) + 0.5 * u2))).mean((0, 1)))
    assert np.isfinite(want["fconm"]).sum() >= 3
    for k, w in want.items():
        assert np.array_equal(np.isnan(got[k]), np.isnan(w)), k
        inf = np.isinf(w)
        assert np.array_equal(np.isinf(got[k]), inf) and np.array_equal(got[k][inf], w[inf]), k
