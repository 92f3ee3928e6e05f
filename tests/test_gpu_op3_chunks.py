"""The drop-in adjoint with its histories passing in chunks of levels: sizes
below and above the threaded path, a level count that leaves a short last
chunk, the smallest histories, in place and into other arrays, against the
FP64 oracle and bit for bit against the allocation-free form, which moves one
level at a time."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _inputs(nz, nx, nt, seed):
    rng = np.random.default_rng(seed)
    hist = [np.asfortranarray(rng.uniform(-1, 1, (nz, nx, nt)), np.float32) for _ in range(5)]
    m1 = [np.asfortranarray(rng.uniform(0.4e-7, 0.6e-7, (nz, nx)), np.float32) for _ in range(2)]
    aux = [np.asfortranarray(rng.uniform(0.5e6, 2.0e6, (nz, nx)), np.float32) for _ in range(3)]
    return hist, m1 + aux


@pytest.mark.parametrize("nz,nx,nt", [(12, 12, 3), (12, 13, 4), (30, 40, 9), (70, 93, 300), (130, 170, 64), (200, 333, 41)])
def test_chunks_equal_single_levels(hip, nz, nx, nt):
    print("op3 chunks", nz, nx, nt, 20 * nz * nx * nt / 2**20, "MiB", flush=True)
    hist, coefs = _inputs(nz, nx, nt, nt)
    keep = [a.copy(order="F") for a in hist]
    want = hip.rtm_op3_noalloc(hist, coefs)
    got = hip.rtm_op3(hist, coefs)
    for f in range(5):
        assert np.array_equal(hist[f], keep[f])  # the input is left alone
        assert np.array_equal(got[f], want[f])
        assert got[f].flags.f_contiguous
    hip.rtm_op3(hist, coefs, inplace=True)
    for f in range(5):
        assert np.array_equal(hist[f], want[f])


def test_short_histories_are_copied(hip):
    hist, coefs = _inputs(20, 20, 2, 1)
    got = hip.rtm_op3(hist, coefs)
    for f in range(5):
        assert np.array_equal(got[f], hist[f]) and got[f] is not hist[f]


def test_chunked_vs_fp64(hip):
    nz, nx, nt = 100, 120, 80
    hist, coefs = _inputs(nz, nx, nt, 7)
    got = hip.rtm_op3(hist, coefs)
    ref = O.rtm_op3_c([a.astype(np.float64) for a in hist], [c.astype(np.float64) for c in coefs])
    for g, r in zip(got, ref):
        assert O.rel_l2(g, r) <= 1e-5
