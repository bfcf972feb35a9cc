"""Downloads of one field of exactly 1 MiB, the most that takes the runtime's own
copy into pageable memory, and of one plane more, which goes through the ring."""

import numpy as np
import pytest

import helpers as H
from test_gpu_download import _box, _check

pytestmark = pytest.mark.gpu

SIZES = [(62, 62, 30), (62, 62, 31)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_one_field_comes_back(size):
    meta, st = _box(size, 7)
    assert (st["rw"].nbytes > 1 << 20) == (size == SIZES[1])
    with H.pkg().Box(meta) as box:
        box.upload(st)
        for k in ("rw", "bz"):
            out = np.zeros_like(st[k])
            ptr = [H.pkg()._ptr(out) if f == k else None for f in H.FIELDS]
            assert box.lib.mhd_download(box.h, *ptr) == 0
            _check({k: out}, st, [k])
