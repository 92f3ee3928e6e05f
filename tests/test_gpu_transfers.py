"""Transfers between host and device on the ways that ordinary sizes do not take:
without the device scratch (as where memory is short), a stacked image beyond the
scratch, and records beyond the size at which several threads copy. All exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(nz, nx, seed):
    rng = np.random.default_rng(seed)
    coefs = [np.asfortranarray(c * rng.uniform(0.5, 1.0, (nz, nx)), np.float32) for c in (1e-7, 1e-7, 1e6, 1e6, 3e6)]
    return coefs, rng


@pytest.mark.parametrize("nz,nx,nt", [(12, 12, 5), (33, 70, 20), (97, 45, 31)])
def test_without_scratch(hip, monkeypatch, nz, nx, nt):
    print("without scratch", nz, nx, nt, flush=True)
    coefs, rng = _model(nz, nx, nt)
    wav = rng.standard_normal(nt).astype(np.float32)
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, nx // 2, nz // 2, nz // 3, 1, nx - 2)
    rec = rng.standard_normal((5, nx - 2, nt)).astype(np.float32)
    dm = [np.asfortranarray(rng.uniform(-1, 1, (nz, nx)), np.float32) for _ in range(3)]
    spec = dict(nz=nz, nx=nx, xs=nx // 2, zs=nz // 2, zr=nz // 3, rx0=1, nrx=nx - 2, img_z0=1, img_x0=2, img_nz=nz - 3,
                img_nx=nx - 2, stack_z0=2, stack_x0=1)

    def run():
        b = hip.Batch(nt, 10.0, 1e-3, [spec] * 2, [coefs] * 2, wav, txr=2, stack_shape=(nz, nx))
        b.set_data(0, rec)
        b.set_data(1, -rec)
        back = [b.get_data(i) for i in range(2)]
        assert np.array_equal(back[0], rec) and np.array_equal(back[1], -rec)
        b.migrate()
        out = [a for i in range(2) for a in b.image(i)] + list(b.stack((nz, nx)))
        b.close()
        r, last = hip.forward(s, coefs, wav, want_last=True)
        return out + [r, *last, hip.born(s, coefs, wav, dm), *hip.migrate(s, coefs, wav, rec)]

    want = run()
    monkeypatch.setenv("RTM_SCRATCH", "0")
    got = run()
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    assert sum(np.abs(w).max() > 0 for w in want) > len(want) // 2


def test_non_finite_results_are_reported_without_scratch(hip, monkeypatch):
    nz, nx, nt = 40, 50, 60
    monkeypatch.setenv("RTM_SCRATCH", "0")
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, 25, 20, 20, 0, nx)
    coefs = [np.full((nz, nx), c * 1e3, np.float32, order="F") for c in (5e-8, 5e-8, 3e5, 3e5, 9e5)]
    with pytest.raises(hip.RtmError) as e:
        hip.forward(s, coefs, np.full(nt, 1e30, np.float32))
    assert e.value.code == -4 and "receiver data" in str(e.value)


# 8.4 million values fill the 32 MiB scratch
@pytest.mark.parametrize("shape", [(1671, 1677), (1700, 3400)])
def test_stack_in_pieces(hip, shape):
    nz, nx, nt = 60, 70, 24
    print("stack", shape, flush=True)
    coefs, rng = _model(nz, nx, 5)
    wav = rng.standard_normal(nt).astype(np.float32)
    corners = [(0, 0), (shape[0] - nz, shape[1] - nx), (shape[0] // 2, 7), (shape[0] // 3, shape[1] - nx)]
    specs = [dict(nz=nz, nx=nx, xs=nx // 2, zs=nz // 2, zr=20, rx0=1, nrx=nx - 2, img_z0=0, img_x0=0, img_nz=nz, img_nx=nx,
                  stack_z0=z, stack_x0=x) for z, x in corners]
    b = hip.Batch(nt, 10.0, 1e-3, specs, [coefs] * 4, wav, txr=2, stack_shape=shape)
    for i in range(4):
        b.set_data(i, rng.standard_normal((5, nx - 2, nt)).astype(np.float32))
    b.migrate()
    want = [np.zeros(shape, np.float32) for _ in range(3)]
    for i, (z, x) in enumerate(corners):
        for w, a in zip(want, b.image(i)):
            w[z:z + nz, x:x + nx] = a
    for g, w in zip(b.stack(shape), want):
        assert np.array_equal(g, w) and np.count_nonzero(w) > nz * nx
    b.close()


# 96 MiB and more go to the device from several threads, in pieces of 4 MiB
@pytest.mark.parametrize("n2,n3,nt", [(131, 127, 1601), (64, 128, 3072)])
def test_large_records(hip, n2, n3, nt):
    print("large record", n2, n3, nt, 4 * n2 * n3 * nt / 2**20, "MiB", flush=True)
    g = hip.Acoustic3D(np.full((11, n2, n3), 0.08, np.float32, order="F"), np.zeros(nt, np.float32), (5, 20, 20), 5, abc=0,
                       snap_every=nt, snap_prec="fp32")
    rec = np.random.default_rng(nt).standard_normal((nt, n3, n2), dtype=np.float32)
    g.set_data(rec)
    assert np.array_equal(g.data(), rec)
    g.close()
