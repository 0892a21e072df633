"""Gradient limiting against the sequential sweeps, bit for bit: one thread's
chain and the segments swept side by side round alike."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    from seismicmesh_amd import _lib
    _lib.require_gpu()


def _sweeps(f, step):
    # forward and backward along each axis in turn, as rounded in FP64
    f = f.copy()
    for ax in range(f.ndim):
        g = np.moveaxis(f, ax, 0)
        with np.errstate(invalid="ignore"):
            for j in range(1, len(g)):
                lim = g[j - 1] + step
                g[j] = np.where(g[j] > lim, lim, g[j])
            for j in range(len(g) - 2, -1, -1):
                lim = g[j + 1] + step
                g[j] = np.where(g[j] > lim, lim, g[j])
    return f


# segment edges (16 values), the row and column tiles, lines of 1, 2 and
# one past the longest held in LDS, an axis of one value
@pytest.mark.parametrize("shape", [
    (1, 1, 1), (2, 1, 1), (1, 17, 1), (15, 16, 1), (33, 65, 1), (129, 700, 1), (700, 129, 1),
    (9300, 3, 1), (3, 9300, 1), (16384, 2, 1), (16385, 2, 1), (2, 16385, 1), (5, 6, 7),
    (31, 40, 77), (64, 1, 130), (1, 50, 60),
    # rows: one thread a line up to 10 values, and up to 64 of 2 M values in all
    (10, 460, 460), (11, 460, 460), (11, 500, 381), (64, 20, 30), (65, 20, 30),
    # more lines than 65535 along axis 0, more planes than that along axis 1
    (20, 260, 260), (70, 256, 257), (2, 3, 65536)])
@pytest.mark.parametrize("kind", ["steps", "ramp", "special"])
def test_limgrad_bit_for_bit(shape, kind):
    import torch
    from seismicmesh_amd import _lib
    rng = np.random.default_rng(sum(shape))
    f = rng.uniform(50.0, 60.0, shape)
    f[rng.random(shape) < 0.02] += 300.0
    if kind == "ramp":
        # one low corner limits whole lines
        f = f + 1e6
        f[0, 0, 0] = 1.0
    elif kind == "special":
        f[rng.random(shape) < 0.01] = np.inf
        f[rng.random(shape) < 0.01] = np.nan
        f[rng.random(shape) < 0.01] = -np.inf
    d = torch.from_numpy(f.ravel(order="F").copy()).cuda()
    _lib.check(_lib.lib.sm_limgrad(ctypes.c_void_p(d.data_ptr()), *shape, 6.28, 0.15, None),
               "sm_limgrad")
    got = d.cpu().numpy().reshape(shape, order="F")
    assert np.array_equal(got, _sweeps(f, 6.28 * 0.15), equal_nan=True)
