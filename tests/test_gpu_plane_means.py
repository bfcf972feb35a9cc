"""The plane means' sequential sums, which a wavefront forms a block of 64 or
512 values at a time: right-hand sides (density diffusion and Rempel conduction
read the means of RO and TT) against the oracle bit for bit, at slabs around the
block sizes and with values that make a block fall back: halfway cases, decades
of magnitude (the binade moves), both signs and cancellation."""

import numpy as np
import pytest

import helpers as H
from test_gpu_parity import random_box

pytestmark = pytest.mark.gpu

SIZES = [(7, 3, 1), (16, 4, 1), (13, 5, 1), (64, 8, 1), (57, 9, 1), (32, 36, 4), (96, 96, 1)]  # npx, npy, npey


def _values(kind, shape, rng):
    if kind == "halves":
        return 1.0 + rng.integers(0, 2**44, shape) * 2.0**-44
    if kind == "decades":
        return 10.0 ** rng.uniform(-6, 6, shape)
    if kind == "constant":
        return np.full(shape, 0.7)
    return rng.standard_normal(shape)  # signs


@pytest.mark.parametrize("lrem", [False, True], ids=["id", "id_lrem"])
@pytest.mark.parametrize("kind", ["halves", "decades", "constant", "signs"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_means_equal_the_sequential_sums(size, kind, lrem):
    npx, npy, npey = size
    meta, st = random_box(npx, npy, 6, lmag=False, lrot=False, seed=npx)
    meta.update(dict(id=1, dh=0.02, dv=0.03, npey=npey))
    if lrem:
        meta.update(dict(lrem=1, itc=1, tu=0.9, dztu=1e-3, dztb=-2e-3, zmax=1.0))
    rng = np.random.default_rng(npx * npy)
    inner = (npx, npy, 8)
    st["tt"][1:-1, 1:-1, :] = _values(kind, inner, rng)
    # (RO keeps one sign: its mean divides)
    st["ro"][1:-1, 1:-1, :] = np.abs(_values(kind, inner, rng)) + 2.0**-10
    for k in ("ro", "tt"):
        H.ics().periodic_fill(st[k])
    o = H.oracle_mod().Oracle(meta, st)
    o.fluxes()
    with H.pkg().Box(meta) as box:
        box.upload(st)
        f = box.fluxes()
    for k in ("fu", "fv", "fw", "fr", "ft"):
        assert np.array_equal(f[k][1:-1, 1:-1, 1:-1], o.arrays[k][1:-1, 1:-1, 1:-1]), k
