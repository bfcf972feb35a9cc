"""Stage launches at the edges of their split: chunks of three planes at the
boundaries (which also apply the boundary conditions), column tiles that do
and do not divide over the XCDs, and work tables whose requested chunk depth
is below three planes.  The FP64 form against the oracle, bit for bit; the
ensemble, whose table splits the planes differently, against single boxes."""

import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


def _box(npx, npy, npz, lmag, seed=3):
    import importlib
    wl = importlib.import_module("rast-3dmhd_amd.workload")
    meta, st = wl.convection_box(npx, npy, npz, seed=seed, lmag=lmag, contrast=5.0, ra=1e4, pm=1.0, ta=1e4, kmax=2)
    rng = np.random.default_rng(seed)
    for k in ("ru", "rv", "rw"):  # a flow, so that every term of the right-hand side counts
        st[k][1:-1, 1:-1, 1:-1] = 0.05 * rng.standard_normal((npx, npy, npz))
        H.ics().periodic_fill(st[k])
    return meta, st


# at most npz - 4 chunks (the first and the last hold three planes); 64x32 has 8 tiles, 130x33 27, 200x16 16
SIZES = [(9, 6, 4), (64, 32, 5), (64, 32, 6), (64, 32, 7), (130, 33, 10), (200, 16, 23), (66, 5, 33)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("lmag", [True, False], ids=["mhd", "hydro"])
def test_fp64_steps_match_the_oracle_at_split_edges(size, lmag):
    meta, st = _box(*size, lmag)
    o = H.oracle_mod().Oracle(meta, st)
    with H.pkg().Box(meta) as box:
        box.upload(st)
        for _ in range(2):
            o.step()
            assert box.step() == (o.meta["dt"], o.meta["umach"])
        got = box.download()
    for k in H.FIELDS[:8 if lmag else 5]:
        assert np.array_equal(got[k], o.arrays[k]), k


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kdepth", [1, 3, 4, 0])
def test_ensemble_chunks_match_single_boxes(precision, kdepth):
    boxes = [_box(*s, True, seed=7 + i) for i, s in enumerate(SIZES)]
    want = []
    for m, s in boxes:
        with H.pkg().Box(m, precision=precision) as box:
            box.upload(s)
            want.append((*box.steps(3), box.clock(), box.download()))
    with H.pkg().Ensemble([m for m, _ in boxes], precision=precision) as ens:
        for b, (_, s) in enumerate(boxes):
            ens.upload(b, s)
        ens.set_tiling(4, kdepth, 5)
        dt, um = ens.steps(3)
        for b, (d, u, clk, ref) in enumerate(want):
            assert (dt[b], um[b], ens.clock(b)) == (d, u, clk), b
            got = ens.download(b)
            for k in H.FIELDS:
                assert np.array_equal(got[k], ref[k]), (b, k)
