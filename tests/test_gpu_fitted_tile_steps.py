"""Boxes large enough that the rules give them fitted tiles (test_host_tile_rules)
against 64x8 tiles of the same box, bit for bit."""

import numpy as np
import pytest

import helpers as H
from test_gpu_stage_split import _box
from test_host_tile_rules import FITTED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [b for b, _ in FITTED], ids=lambda b: "x".join(map(str, b)))
def test_fitted_steps_match_64x8(box, monkeypatch):
    npx, npy, npz, lmag, precision, diffusion = box
    meta, st = _box(npx, npy, npz, lmag)
    if diffusion:
        meta.update(dict(id=1, dh=0.02, dv=0.03))

    def run():
        with H.pkg().Box(meta, precision=precision) as b:
            b.upload(st)
            f = b.fluxes() if precision == "fp64" else {}
            return b.steps(2), b.download(), f

    got = run()
    monkeypatch.setenv("RAST3DMHD_TILE_Y", "8")
    want = run()
    assert got[0] == want[0]
    for g, w in zip(got[1:], want[1:]):
        for k in w:
            if lmag or k not in ("bx", "by", "bz", "ww1", "ww2", "ww3"):
                assert np.array_equal(g[k], w[k]), k
