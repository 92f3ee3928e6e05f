"""The eight-wave tile of width 1 (64 x 8 cells, one per thread, fp32
snapshots) against width 2's bit for bit: grids at the edges of the tile and
the smallest one, every adjoint sponge, imaging with the full history and
decimated, Born modelling with its sources formed in the step, the drop-in
adjoint, and a batch of uneven shots (tile table instead of tile numbers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(12, 12), (64, 8 * 4), (65, 33), (63, 15), (128, 24), (90, 107)]


def _model(nz, nx, seed):
    rng = np.random.default_rng(seed)
    return [np.asfortranarray(c * rng.uniform(0.5, 1.0, (nz, nx)), np.float32)
            for c in (1e-7, 1e-7, 1e6, 1e6, 3e6)], rng


def _both(monkeypatch, fn):
    out = []
    for txr in ("1", "2"):
        monkeypatch.setenv("RTM_TXR", txr)
        out.append(fn())
    monkeypatch.delenv("RTM_TXR")
    out.append(fn())  # the default of single-shot calls
    return out


def _same(outs):
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            assert np.array_equal(a, b) and np.isfinite(a).all()
    assert max(np.abs(a).max() for a in outs[0]) > 0


@pytest.mark.parametrize("nz,nx", GRIDS)
@pytest.mark.parametrize("adj_abc,every,comp", [(0, 1, 0), (1, 1, 1), (2, 1, 0), (1, 3, 1)])
def test_migration(hip, monkeypatch, nz, nx, adj_abc, every, comp):
    print("width 1 migration", nz, nx, adj_abc, every, flush=True)
    nt, abc = 40, 6 if min(nz, nx) > 22 else 0
    coefs, rng = _model(nz, nx, nz + nx)
    rec = rng.standard_normal((5, nx - 3, nt)).astype(np.float32)
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, nx // 2, nz // 2, nz // 3, 2, nx - 3, abc, adj_abc=adj_abc, snap_every=every,
                 comp_image=comp)
    wav = rng.standard_normal(nt).astype(np.float32)
    _same(_both(monkeypatch, lambda: hip.migrate(s, coefs, wav, rec)))


@pytest.mark.parametrize("nz,nx", GRIDS)
def test_born_and_record(hip, monkeypatch, nz, nx):
    print("width 1 Born", nz, nx, flush=True)
    nt, abc = 30, 6 if min(nz, nx) > 22 else 0
    coefs, rng = _model(nz, nx, 3 * nz + nx)
    dm = [np.asfortranarray(rng.uniform(-1, 1, (nz, nx)), np.float32) for _ in range(3)]
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, nx // 2, nz // 2, nz // 3, 0, nx, abc)
    wav = rng.standard_normal(nt).astype(np.float32)
    _same(_both(monkeypatch, lambda: [hip.born(s, coefs, wav, dm), hip.forward(s, coefs, wav)]))
    # the marching forward takes the sources from a buffer of their own
    a = hip.born(s, coefs, wav, dm)
    monkeypatch.setenv("RTM_TBLOCK", "2")
    monkeypatch.setenv("RTM_MARCH_W", "16")
    assert np.array_equal(a, hip.born(s, coefs, wav, dm))


@pytest.mark.parametrize("nz,nx", GRIDS)
def test_drop_in(hip, monkeypatch, nz, nx):
    print("width 1 drop-in", nz, nx, flush=True)
    coefs, rng = _model(nz, nx, 7 * nz + nx)
    hist = [np.asfortranarray(rng.standard_normal((nz, nx, 9)), np.float32) for _ in range(5)]
    _same(_both(monkeypatch, lambda: hip.rtm_op3(hist, coefs)))


def test_uneven_batch(hip):
    nt, shots, coefs, recs = 30, [], [], []
    for k, (nz, nx) in enumerate([(70, 90), (64, 41), (129, 64)]):
        c, rng = _model(nz, nx, k)
        coefs.append(c)
        shots.append(dict(nz=nz, nx=nx, xs=nx // 2, zs=nz // 2, zr=nz // 3, rx0=1, nrx=nx - 2))
        recs.append(rng.standard_normal((5, nx - 2, nt)).astype(np.float32))
    wav = np.random.default_rng(9).standard_normal(nt).astype(np.float32)
    imgs = []
    for txr in (1, 2):
        b = hip.Batch(nt, 10.0, 1e-3, shots, coefs, wav, abc=5, adj_abc=1, txr=txr)
        for i, r in enumerate(recs):
            b.set_data(i, r)
        b.migrate()
        imgs.append([a for i in range(3) for a in b.image(i)])
        b.close()
    _same(imgs)


@pytest.mark.parametrize("prec", ["bf16", "fp16"])
def test_tuner_keeps_the_scales_of_width_2(hip, prec):
    """16-bit snapshots are scaled per strip of the tile width: a tuned batch
    gives the images of width 2 bit for bit."""
    nz, nx, nt = 70, 90, 24
    c, rng = _model(nz, nx, 3)
    spec = dict(nz=nz, nx=nx, xs=45, zs=30, zr=20, rx0=1, nrx=nx - 2)
    rec = rng.standard_normal((5, nx - 2, nt)).astype(np.float32)
    wav = rng.standard_normal(nt).astype(np.float32)
    imgs = []
    for txr in (0, 2):
        b = hip.Batch(nt, 10.0, 1e-3, [spec], [c], wav, abc=5, adj_abc=1, snap_every=3, snap_prec=prec, comp_image=1,
                      txr=txr)
        assert b.txr == 2
        b.set_data(0, rec)
        b.migrate()
        imgs.append(list(b.image(0)))
        b.close()
    _same(imgs)
