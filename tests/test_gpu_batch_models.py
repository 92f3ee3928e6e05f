"""Batches whose settings change between runs. The true model is set again between
syntheses: the second data set is that of the second model, also when the
launches are replayed from graphs captured with the first one, with one and
with several shots a group and with one and two levels a launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pair", ["0", "1"])
@pytest.mark.parametrize("shots", [1, 2])
def test_true_model_set_again(hip, monkeypatch, shots, pair):
    nz, nx, nt = 61, 77, 33
    monkeypatch.setenv("RTM_PAIR", pair)
    rng = np.random.default_rng(shots)
    coefs = [np.asfortranarray(c * rng.uniform(0.5, 1.0, (nz, nx)), np.float32) for c in (1e-7, 1e-7, 1e6, 1e6, 3e6)]
    models = [[np.asfortranarray(c * np.float32(f)) for c in coefs] for f in (1.05, 0.9, 1.02)]
    wav = rng.standard_normal(nt).astype(np.float32)
    spec = dict(nz=nz, nx=nx, xs=nx // 2, zs=nz // 2, zr=20, rx0=1, nrx=nx - 2)

    def batch(graph):
        return hip.Batch(nt, 10.0, 1e-3, [spec] * shots, [coefs] * shots, wav, abc=6, adj_abc=1, txr=1, use_graph=graph)

    def data(b, model):
        b.set_true_model([model] * shots)
        b.synthesize()
        return [b.get_data(i) for i in range(shots)]

    kept = batch(1)
    for model in models:
        print("true model again", shots, pair, flush=True)
        fresh = batch(0)
        want = data(fresh, model)
        fresh.close()
        for g, w in zip(data(kept, model), want):
            assert np.array_equal(g, w) and np.abs(w).max() > 0
    kept.close()


@pytest.mark.parametrize("created,run", [("-1", "0"), ("0", "-1"), ("3", "0"), ("0", "3")])
def test_levels_a_launch_are_the_batchs_own(hip, monkeypatch, created, run):
    """How many levels a launch takes, and with it the ring of levels, is decided
    when a batch is created: a run under another RTM_PAIR (-1: the rule) gives the
    same images."""
    nz, nx = 61, 77
    spec = dict(nz=nz, nx=nx, xs=nx // 2, zs=nz // 2, zr=20, rx0=1, nrx=nx - 2)
    rng = np.random.default_rng(3)
    coefs = [np.asfortranarray(c * rng.uniform(0.5, 1.0, (nz, nx)), np.float32) for c in (1e-7, 1e-7, 1e6, 1e6, 3e6)]
    for nt in (32, 33, 34, 35):
        print("levels a launch", created, run, nt, flush=True)
        rec = rng.standard_normal((5, nx - 2, nt)).astype(np.float32)
        wav = rng.standard_normal(nt).astype(np.float32)
        monkeypatch.setenv("RTM_PAIR", created)
        b = hip.Batch(nt, 10.0, 1e-3, [spec], [coefs], wav, abc=6, adj_abc=1, txr=1)
        b.set_data(0, rec)
        b.migrate()
        want = b.image(0)
        monkeypatch.setenv("RTM_PAIR", run)
        b.migrate()
        for w, g in zip(want, b.image(0)):
            assert np.array_equal(g, w) and np.abs(w).max() > 0
        b.close()


@pytest.mark.parametrize("nx,form", [(10355, 2), (10357, 0)])
def test_reported_form_of_large_grids(hip, monkeypatch, nx, form):
    """The marching forms take grids of up to 2^31 / 20 cells (columns of 10368
    rows: 10356); a batch that asked for one on a larger grid says that it runs
    tiles."""
    nz = 10368
    print("large grid", nz, nx, flush=True)
    monkeypatch.setenv("RTM_TBLOCK", "2")
    field = np.zeros((nz, nx), np.float32, order="F")
    spec = dict(nz=nz, nx=nx, xs=20, zs=20, zr=20, rx0=0, nrx=4)
    b = hip.Batch(2, 10.0, 1e-3, [spec], [[field] * 5], np.ones(2, np.float32), txr=2, snap_every=2)
    assert b.tblock == form
    b.close()
