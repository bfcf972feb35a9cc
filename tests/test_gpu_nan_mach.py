"""A NaN in the state, of either sign, shows in UMACH of the step that starts from
it, whether the stand-alone reduction or the step before formed it."""

import ctypes as C

import numpy as np
import pytest

import helpers as H
from test_gpu_stage_split import _box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nan", [np.nan, -np.nan], ids=["+", "-"])
@pytest.mark.parametrize("field", ["ru", "ro", "tt"])
@pytest.mark.parametrize("lmag", [True, False], ids=["mhd", "hydro"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_nan_reaches_umach(precision, lmag, field, nan):
    meta, st = _box(20, 9, 8, lmag)
    clean = {k: a.copy(order="F") for k, a in st.items()}
    st[field][7, 5, 4] = nan
    with H.pkg().Box(meta, precision=precision) as box:
        if precision == "mixed":  # (the mean planes of a state with a NaN are no background)
            box.set_background(*H.pkg()._horizontal_means(clean))
        box.upload(st)
        for _ in range(2):
            dt, um = C.c_double(0.0), C.c_double(0.0)
            assert box.lib.mhd_step(box.h, C.byref(dt), C.byref(um)) == H.pkg().MHD_ERR_NONFINITE
            assert np.isnan(um.value)
