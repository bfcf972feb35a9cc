"""Weight gradients of one infinite output gradient: infinite, with the sign of
the activation it multiplies, for every tap inside the volume; finite for the
other channels; on rows that do and do not fill the weight gradient's segments of
64 voxels.  (An activation below the rounding of the GELU is a zero there, and
its product a NaN: activations are compared from 0.1 on.)"""

import os
import sys

import numpy as np
import pytest

import helpers as H

sys.path.insert(0, os.path.join(H.REPO, "oracle"))
import net_oracle as N  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 8), (64, 6, 4), (70, 5, 6), (33, 9, 4), (3, 4, 5)], ids=lambda s: "x".join(map(str, s)))
def test_one_infinite_gradient(shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(4)
    net = H.pkg().Net(8, 32, 7)
    sizes = [32 * 27 * 8, 32, 32 * 27 * 32, 32, 7 * 27 * 32, 7]
    vec = (0.1 * rng.standard_normal(sum(sizes))).astype(np.float32)
    net.set_params(vec)
    x = rng.standard_normal((nz, ny, nx, 8)).astype(np.float32)
    dy = rng.standard_normal((nz, ny, nx, 7)).astype(np.float32)
    dy[nz - 1, 0, nx - 1, 5] = np.inf
    g = net.gradient(x, dy)
    net.close()
    off = np.cumsum([0] + sizes)
    w3, b3 = g[off[4]:off[5]].reshape(7, 27, 32), g[off[5]:]
    o = N.Net(N.unflatten(vec, 8, 32, 7), bf16_emulation=True)
    o.forward(x, keep=True)
    # (the taps of dz = +1 multiply the infinity by the zeros below the last plane)
    a2 = np.stack([N.shift(o.cache[4], *tap)[nz - 1, 0, nx - 1] for tap in N.TAPS[:18]])
    sure = np.abs(a2) > 0.1
    assert sure.mean() > 0.4
    assert np.array_equal(w3[5, :18][sure], np.inf * a2[sure]) and np.isinf(b3[5])
    others = [0, 1, 2, 3, 4, 6]
    assert np.isfinite(w3[others]).all() and np.isfinite(b3[others]).all()
