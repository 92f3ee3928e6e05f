"""Rearrangement of records and fields between the callers' layouts and the
device's (exact copies): odd sizes around the 64 x 64 transpose tile, single
traces and samples, and arrays beyond the 32 MiB device scratch, which go
through it in pieces."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _coefs(nz, nx, v=1.0):
    return [np.full((nz, nx), c * v, np.float32, order="F") for c in (5e-8, 5e-8, 3e5, 3e5, 9e5)]


@pytest.mark.parametrize("nt,nrx", [(1, 1), (3, 64), (64, 63), (65, 1), (129, 65), (3000, 700)])
def test_records_come_back_as_they_were_set(hip, nt, nrx):
    nz, nx = 20, max(nrx, 12) + 3
    print("records", nt, nrx, flush=True)
    spec = dict(nz=nz, nx=nx, xs=nx // 2, zs=8, zr=9, rx0=2, nrx=nrx)
    b = hip.Batch(nt, 10.0, 1e-3, [spec, spec], [_coefs(nz, nx)] * 2, np.zeros(nt, np.float32), txr=2)
    rng = np.random.default_rng(nt + nrx)
    recs = [rng.standard_normal((5, nrx, nt)).astype(np.float32) for _ in range(2)]
    for i, r in enumerate(recs):
        b.set_data(i, r)
    for i, r in enumerate(recs):
        assert np.array_equal(b.get_data(i), r)
    b.close()


# the last levels (unpadded on the device) against the movie's windows (pitched
# copies): 5 fields of 1300 x 1300 exceed the scratch
@pytest.mark.parametrize("nz,nx", [(12, 12), (33, 70), (64, 64), (97, 45), (1300, 1300)])
def test_last_levels_equal_movie_frames(hip, nz, nx):
    nt = 24
    print("fields", nz, nx, flush=True)
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, nx // 2, nz // 2, nz // 2, 0, nx)
    wav = np.ones(nt, np.float32)
    rng = np.random.default_rng(nz)
    coefs = [np.asfortranarray(c * rng.uniform(0.5, 1.0, (nz, nx)), np.float32) for c in _coefs(nz, nx)]
    rec, last = hip.forward(s, coefs, wav, want_last=True)
    movie, every = hip.forward_movie(s, coefs, wav, nt, 0, 0, nz, nx)
    assert every == 1 and np.abs(last[5]).max() > 0
    for lv in range(2):
        for f in range(5):
            assert np.array_equal(last[5 * lv + f], movie[nt - 2 + lv][f])
    # the record is row zr of every level
    assert np.array_equal(rec[0], np.stack([m[0][nz // 2] for m in movie], 1))


def test_non_finite_results_are_still_reported(hip):
    nz, nx, nt = 40, 50, 60
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, 25, 20, 20, 0, nx)
    with pytest.raises(hip.RtmError) as e:
        hip.forward(s, _coefs(nz, nx, 1e3), np.full(nt, 1e30, np.float32))
    assert e.value.code == -4 and "receiver data" in str(e.value)
