"""Two levels per launch on small grids (elastic2d_pair.hip) against one level
per launch bit for bit: every tile, at the edges of the tiles and on the
smallest grid, odd and even numbers of levels, every snapshot form the pair
kernels write or read, the adjoint sponges, Born modelling, records and the
last levels; and the rule that chooses the tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = ["1", "2", "3", "4"]  # S 22 x 6, M 22 x 14, L 22 x 22, X 54 x 22 (forward)
GRIDS = [(12, 12), (22, 22), (23, 45), (54, 67), (109, 44), (130, 15)]


def _setup(hip, nz, nx, nt, **kw):
    rng = np.random.default_rng(nz + 3 * nx + nt)
    coefs = [np.asfortranarray(c * rng.uniform(0.5, 1.0, (nz, nx)), np.float32) for c in (1e-7, 1e-7, 1e6, 1e6, 3e6)]
    s = hip.shot(nz, nx, nt, 10.0, 1e-3, nx // 2, nz // 2, nz // 3, 2, nx - 3, 6 if min(nz, nx) > 22 else 0, **kw)
    wav = rng.standard_normal(nt).astype(np.float32)
    return s, coefs, wav, rng


def _same(monkeypatch, tile, fn):
    outs = []
    for t in ("0", tile):
        monkeypatch.setenv("RTM_PAIR", t)
        outs.append(fn())
    for a, b in zip(*outs):
        assert np.array_equal(a, b) and np.isfinite(a).all()
    assert max(np.abs(a).max() for a in outs[0]) > 0


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("nz,nx", GRIDS)
def test_pairs(hip, monkeypatch, nz, nx, tile):
    for nt, adj_abc, every, comp in ((31, 0, 1, 0), (30, 1, 1, 1), (31, 2, 1, 0), (30, 1, 2, 0), (32, 1, 3, 1)):
        print("pairs", tile, nz, nx, nt, adj_abc, every, flush=True)
        s, coefs, wav, rng = _setup(hip, nz, nx, nt, adj_abc=adj_abc, snap_every=every, comp_image=comp)
        rec = rng.standard_normal((5, nx - 3, nt)).astype(np.float32)
        dm = [np.asfortranarray(rng.uniform(-1, 1, (nz, nx)), np.float32) for _ in range(3)]
        _same(monkeypatch, tile, lambda: hip.migrate(s, coefs, wav, rec))
        _same(monkeypatch, tile, lambda: hip.forward(s, coefs, wav, want_last=True))
        if every == 1:
            _same(monkeypatch, tile, lambda: [hip.born(s, coefs, wav, dm)])


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("tile", TILES)
def test_one_shot_batch(hip, monkeypatch, tile, graph):
    """Synthesized data (the second run subtracts from the record) and migrations
    of a one-shot batch, twice, the second time from the captured graphs."""
    nz, nx, nt = 61, 77, 33
    s, coefs, wav, rng = _setup(hip, nz, nx, nt)
    true = [np.asfortranarray(c * np.float32(1.05)) for c in coefs]
    spec = dict(nz=nz, nx=nx, xs=nx // 2, zs=nz // 2, zr=20, rx0=1, nrx=nx - 2)

    def run():
        b = hip.Batch(nt, 10.0, 1e-3, [spec], [coefs], wav, abc=6, adj_abc=1, txr=1, use_graph=graph)
        b.set_true_model([true])
        out = []
        for _ in range(2):
            b.synthesize()
            out.append(b.get_data(0))
            b.migrate()
            out += list(b.image(0))
        b.close()
        return out

    _same(monkeypatch, tile, run)


@pytest.mark.parametrize("nt", [1, 2, 3, 4])
def test_few_levels(hip, monkeypatch, nt):
    s, coefs, wav, rng = _setup(hip, 40, 30, nt)
    rec = rng.standard_normal((5, 27, nt)).astype(np.float32)
    outs = []
    for t in ("0", "1"):
        monkeypatch.setenv("RTM_PAIR", t)
        outs.append([*hip.migrate(s, coefs, wav, rec), *hip.forward(s, coefs, wav, want_last=True)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_rule(hip, monkeypatch):
    """Two levels a launch on small grids, one on large ones."""
    nt = 12
    for nz, nx, levels in ((64, 90, 2), (300, 300, 2), (900, 1300, 1)):
        s, coefs, wav, rng = _setup(hip, nz, nx, nt)
        rec = rng.standard_normal((5, nx - 3, nt)).astype(np.float32)
        hip.migrate(s, coefs, wav, rec)
        t = hip.timings()
        # the forward's level 2 goes alone: it has no sponge
        assert (t[1], t[3]) == ((6, 6) if levels == 2 else (nt - 1, nt)), (nz, nx, t)
