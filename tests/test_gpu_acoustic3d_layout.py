"""The padded device layout of the 3D acoustic fields against contiguous rows
(what runs where memory is short), bit for bit: rows that end at, before and
after a multiple of the padding, the snapshots written by the step that reads
their level and the last one by a pass of its own, modelled records, images and
snapshot scales; and the scales against the fields' own maxima (single-precision rounding of 20 levels, 20 x 10 x
6e-8)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _run(hip, c, amp, src, rec, j, prec, abc):
    g = hip.Acoustic3D(c, amp, src, 6, abc=abc, snap_every=j, snap_prec=prec)
    g.model_data(c * np.float32(1.03))
    d = g.data()
    g.set_data(rec)
    g.migrate()
    scales = np.zeros(max(len(amp) // j, 1), np.float32)
    hip.load().ac3d_get_snapshot_scales(g._h, scales.ctypes.data_as(C.c_void_p), C.c_int(scales.size))
    out = [d, g.image(), scales]
    g.close()
    return out


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("shape", [(37, 14, 23), (38, 21, 12), (101, 30, 26), (64, 11, 33)])
@pytest.mark.parametrize("nt,j", [(20, 4), (19, 4), (7, 1), (3, 5)])
def test_padded_rows(hip, monkeypatch, shape, prec, nt, j):
    print("acoustic layout", shape, prec, nt, j, flush=True)
    rng = np.random.default_rng(sum(shape))
    c = np.asfortranarray(rng.uniform(0.06, 0.09, shape), np.float32)
    amp = rng.standard_normal(nt).astype(np.float32)
    src = tuple(n // 2 for n in shape)
    rec = np.zeros((nt, shape[2], shape[1]), np.float32)
    rec[:, 5:-5, 5:-5] = 0.1 * rng.standard_normal((nt, shape[2] - 10, shape[1] - 10))
    abc = 6 if min(shape) >= 22 else 0
    outs = []
    for pad in ("1", "0"):
        monkeypatch.setenv("RTM_AC3_PAD", pad)
        outs.append(_run(hip, c, amp, src, rec, j, prec, abc))
    for a, b in zip(*outs):
        assert np.array_equal(a, b) and np.isfinite(a).all()
    if nt // j:
        # a level spreads a field by 5 cells: with too few the source's and the
        # receivers' never meet and the image is zero
        assert np.abs(outs[0][1]).max() > 0 or 5 * nt < shape[0]
        _, snap = O.ac3_run(c, amp, src, 6, abc=abc, j=j, want_snap=True, nthreads=8)
        top = np.abs(np.asarray(snap, np.float64)).reshape(nt // j, -1).max(axis=1)
        assert np.allclose(outs[0][2][: nt // j], top, rtol=2e-5, atol=0)
