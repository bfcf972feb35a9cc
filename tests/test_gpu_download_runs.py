"""Downloads that come down in runs of up to four pieces (1 MiB and more) without
threads, their pieces cut inside fields: one piece, several, four of more than
1 MiB, and just past the size from which threads take over; some fields left
out.  An uploaded state comes back bit for bit."""

import numpy as np
import pytest

import helpers as H
from test_gpu_download import _box, _check

pytestmark = pytest.mark.gpu

# 8 padded fields: 0.52, 1.06, 3.5, 6.5, 8.3 and 8.5 MB (1 MiB, 8 MiB = 1.05, 8.39 MB)
SIZES = [(19, 17, 18), (22, 23, 26), (37, 33, 38), (45, 47, 42), (49, 50, 47), (49, 50, 48)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_state_comes_back_in_runs(size):
    meta, st = _box(size, 3)
    with H.pkg().Box(meta) as box:
        box.upload(st)
        _check(box.download(), st)
        out = {k: np.zeros_like(st[k]) for k in H.FIELDS[1::2]}
        ptr = [H.pkg()._ptr(out[k]) if k in out else None for k in H.FIELDS]
        assert box.lib.mhd_download(box.h, *ptr) == 0
        _check(out, st, H.FIELDS[1::2])
