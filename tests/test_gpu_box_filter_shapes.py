"""Box filter of the resident state at every read form (factors 2, 4 and 8 in
16-byte pieces, any other point by point) and at the ends of a thread's run of
coarse planes, against the same sums in the same order, bit for bit; mean flux
profiles of planes smaller and larger than their workgroups' shares."""

import numpy as np
import pytest

import helpers as H
from test_gpu_flux_profiles import _compare
from test_gpu_parity import random_box
from test_gpu_stage_split import _box

pytestmark = pytest.mark.gpu

CASES = [(2, 0, (10, 6, 36)), (2, 1, (6, 4, 19)), (3, 0, (9, 6, 30)), (4, 1, (20, 12, 41)), (4, 0, (8, 4, 36)),
         (5, 0, (15, 5, 10)), (6, 1, (12, 6, 61)), (8, 1, (16, 24, 73)), (8, 0, (8, 8, 8)), (1, 0, (5, 7, 9))]


def _filter(a, f, zmode):
    """a[k][j][i], planes 1..npz, summed as the kernel documents it."""
    s = np.zeros((a.shape[0], a.shape[1] // f, a.shape[2] // f))
    for jj in range(f):
        for ii in range(f):
            s = s + a[:, jj::f, ii::f]
    h = s / (f * f)
    if zmode == 0:
        v = np.zeros((a.shape[0] // f,) + h.shape[1:])
        for kk in range(f):
            v = v + h[kk::f]
        return v / f
    nzc = (a.shape[0] - 1) // f + 1
    out = [h[0]]
    for K in range(1, nzc - 1):
        v = 0.0
        for d in range(-(f // 2), f // 2 + 1):
            v = v + (0.5 if abs(d) == f // 2 else 1.0) * h[K * f + d]
        out.append(v / f)
    return np.stack(out + [h[(nzc - 1) * f]])


@pytest.mark.parametrize("factor,zmode,size", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_box_filter_forms(factor, zmode, size):
    meta, st = _box(*size, True)
    with H.pkg().Box(meta) as box:
        box.upload(st)
        got = box.box_filter(factor, zmode, "state")
    for n, k in enumerate(H.FIELDS):
        a = np.ascontiguousarray(np.transpose(st[k][1:-1, 1:-1, 1:-1], (2, 1, 0)))
        assert np.array_equal(got[n], _filter(a, factor, zmode)), k


@pytest.mark.parametrize("shape", [(5, 7, 4), (64, 32, 5), (97, 61, 6)], ids=lambda s: "x".join(map(str, s)))
def test_flux_profiles_at_workgroup_shares(shape):
    meta, st = random_box(*shape, lmag=False, lrot=False, seed=sum(shape))
    o = H.oracle_mod().Oracle(meta, st)
    with H.pkg().Box(meta) as box:
        box.upload(st)
        _compare(box.flux_profiles(), o.flux_profiles(), st)
