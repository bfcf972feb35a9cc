"""Downloads into arrays that the caller pinned: fields just below and above 384
KiB, from which they are copied to directly, a launch per field (more than 16 MiB)
and a run of all fields; one field alone, and a pageable array among them.  An
uploaded state comes back bit for bit."""

import ctypes

import pytest
import torch

import helpers as H
from test_gpu_download import _box, _check

pytestmark = pytest.mark.gpu

# a padded field: 390.7 and 393.7 KB (384 KiB = 393.2 KB), 3.2 and 17.6 MB
SIZES = [(38, 35, 31), (33, 35, 36), (71, 73, 70), (128, 128, 128)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_state_comes_back_in_pinned_arrays(size):
    meta, st = _box(size, 5)

    def fresh(pinned=True):
        return torch.zeros(st["ro"].T.shape, dtype=torch.float64, pin_memory=pinned)

    def get(box, arrays):
        ptr = [ctypes.cast(arrays[k].data_ptr(), H.pkg()._P) if k in arrays else None for k in H.FIELDS]
        assert box.lib.mhd_download(box.h, *ptr) == 0
        _check({k: a.numpy().T for k, a in arrays.items()}, st, arrays)

    with H.pkg().Box(meta) as box:
        box.upload(st)
        get(box, {k: fresh() for k in H.FIELDS})
        get(box, {"ro": fresh()})
        get(box, {k: fresh(k != "by") for k in H.FIELDS[2:7]})
