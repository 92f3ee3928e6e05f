"""The 3D elastic step on the shapes at which its partition changes (one cell
an axis, tiles of 64 rows and a remainder of one, even splits, one plane a
workgroup), against the FP64 oracle at the tolerance of one step (1e-6), and
several steps in a row."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 64, 16), (2, 65, 17), (5, 50, 21), (6, 129, 23), (11, 33, 45), (70, 20, 9)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("steps", [1, 2])
def test_tile_edges_vs_fp64(hip, shape, steps):
    ny, nz, nx = shape
    print("elastic3d tiles", shape, steps, flush=True)
    blocks = [O.el3_random(ny, nz, nx, 41 + s) for s in range(3)]
    coef = O.el3_random(ny, nz, nx, 44, k=6)
    dev = [hip.DeviceArray(b) for b in blocks]
    roles = hip.el3_steps_dev(dev, hip.DeviceArray(coef), steps)
    ref = O.el3_steps(*blocks, coef, steps, nthreads=8)
    for got, want in zip(roles, ref):
        g = got.get()
        for k in range(9):
            assert O.rel_l2(g[k], want[k]) <= 1e-6 * steps
        # the padding is not written
        for ax in range(1, 4):
            for at in (slice(0, 5), slice(-5, None)):
                i = [slice(None)] * 4
                i[ax] = at
                assert not g[tuple(i)].any()
