"""Stage tiles fitted to a box's width against 64x8 tiles (RAST3DMHD_TILE_Y) of
the same box, bit for bit: whole rows as one run, parts of rows, threads past the
tile's last point, rows left over at the bottom and boxes lower than a tile;
right-hand side, steps, density diffusion, and the ensemble's items."""

import numpy as np
import pytest

import helpers as H
from test_gpu_stage_split import _box

pytestmark = pytest.mark.gpu

# FP64: 40x6, 72x3, 40x6, 48x5, 44x5 and 65x3, 33x7; mixed: 40x6, 72x3, 80x3, 48x5, 64x4, 33x7
SIZES = [(40, 13, 9), (72, 10, 6), (80, 25, 7), (96, 11, 5), (130, 90, 8), (33, 65, 6), (17, 4, 6), (88, 3, 5)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("lmag", [True, False], ids=["mhd", "hydro"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_fitted_tiles_match_64x8(size, lmag, precision, monkeypatch):
    meta, st = _box(*size, lmag)
    if precision == "fp64" and size[0] == 96:
        meta.update(dict(id=1, dh=0.02, dv=0.03))

    def run():
        with H.pkg().Box(meta, precision=precision) as box:
            box.upload(st)
            f = box.fluxes() if precision == "fp64" else {}
            return box.steps(3), box.download(), f

    got = run()
    monkeypatch.setenv("RAST3DMHD_TILE_Y", "8")
    want = run()
    assert got[0] == want[0]
    for g, w in zip(got[1:], want[1:]):
        for k in w:
            if lmag or k not in ("bx", "by", "bz", "ww1", "ww2", "ww3"):
                assert np.array_equal(g[k], w[k]), k


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_ensemble_items_match_64x8(precision):
    boxes = [_box(*s, True, seed=11 + i) for i, s in enumerate(SIZES)]
    res = []
    for ty in (4, 8):
        ens = H.pkg().Ensemble([m for m, _ in boxes], precision=precision)
        ens.set_tiling(ty, 4, 0)
        for b, (_, s) in enumerate(boxes):
            ens.upload(b, s)
        out = ens.steps(3)
        res.append((out, [ens.download(b) for b in range(len(boxes))]))
        ens.close()
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)
    for a, b in zip(res[0][1], res[1][1]):
        for k in H.FIELDS:
            assert np.array_equal(a[k], b[k]), k
