"""Mean flux profiles against extended-precision means: the sums carry their
rounding errors, so what is left is the rounding of the terms (12 operations
each at most) and of the last steps."""

import numpy as np
import pytest

import helpers as H
from test_gpu_stage_split import _box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(5, 7, 4), (33, 31, 6), (100, 120, 5)], ids=lambda s: "x".join(map(str, s)))
def test_profiles_are_rounded_means(size):
    meta, st = _box(*size, True)
    with H.pkg().Box(meta) as box:
        box.upload(st)
        got = box.flux_profiles()
    L = np.longdouble
    ru, rv, rw, ro, tt = (st[k][1:-1, 1:-1, 1:-1].astype(L) for k in ("ru", "rv", "rw", "ro", "tt"))
    mean = lambda a: a.mean((0, 1))  # noqa: E731
    w1, uu = tt - mean(tt), (ru**2 + rv**2 + rw**2) / ro**2
    eps = L(2.0) ** -53
    for k, a in (("ttm", tt), ("rom", ro)):
        assert np.all(np.abs(got[k] - mean(a)) <= 3 * eps * mean(np.abs(a))), k
    f = mean(-rw * (L(2.5) * w1 + L(0.5) * uu))
    term = mean(np.abs(rw)) * (5 * np.abs(w1).max((0, 1)) + uu.max((0, 1)))
    assert np.all(np.abs(got["fconm"] - f) <= 12 * eps * term + 3 * eps * np.abs(f))
