"""Network kernels at the edges of their tiles: rows shorter than a tile, one
past one and two tiles, single planes and rows, odd row counts (the weight
gradient takes rows in pairs), against the BF16-emulating oracle with the
tolerances of the full-size comparison (FP32 against FP64 accumulation of
BF16-rounded values: 2e-3 of the RMS forward, 1e-2 for gradients)."""

import os
import sys

import numpy as np
import pytest

import helpers as H

sys.path.insert(0, os.path.join(H.REPO, "oracle"))
import net_oracle as N  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 3), (2, 5, 63), (3, 4, 65), (1, 9, 130), (4, 3, 16), (9, 2, 64), (17, 7, 20)]


def rel(a, b):
    return float(np.sqrt(np.mean((a - b) ** 2)) / np.sqrt(np.mean(b ** 2)))


@pytest.mark.parametrize("cout", [7, 8, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_forward_and_gradients_at_tile_edges(shape, cout):
    nz, ny, nx = shape
    rng = np.random.default_rng(sum(shape))
    p = N.init_params(8, 32, cout, seed=5)
    x = N.bf16(rng.standard_normal((nz, ny, nx, 8)))
    dy = N.bf16(rng.standard_normal((nz, ny, nx, cout)))
    o = N.Net(p, bf16_emulation=True)
    ref = o.forward(x)
    g_ref, dx_ref = o.backward(x, dy)
    with H.pkg().Net(8, 32, cout) as net:
        net.set_params(N.flatten(p))
        y = net.forward(x)
        g, dx = net.gradient(x, dy, want_dx=True)
        g2 = net.gradient(x, dy)
    assert rel(y, ref) <= 2e-3
    got = N.unflatten(g, 8, 32, cout)
    for k in ("W3", "b3", "W2", "b2", "W1", "b1"):
        assert rel(got[k], g_ref[k]) <= 1e-2, k
    assert rel(dx, dx_ref) <= 1e-2
    assert np.array_equal(g, g2)  # fixed-order sums
