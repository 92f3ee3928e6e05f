"""3D acoustic migrations on the shapes at which the step's partition changes
(one interior cell an axis, tile remainders, one plane a workgroup to many),
against the FP64 oracle, and the planes a workgroup marches against each
other bit for bit. Tolerances: single-precision rounding grows by at most a
few units a level, 60 levels x 6e-8 x ~10 operations stays below 1e-4;
bfloat16 snapshots add their own rounding, 2^-9 of each snapshot's maximum."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _case(n1, n2, n3, nt, seed):
    rng = np.random.default_rng(seed)
    c = np.asfortranarray(rng.uniform(0.06, 0.09, (n1, n2, n3)), np.float32)
    t = np.arange(1, nt + 1, dtype=np.float64)
    a = (np.pi * (t - 12.0) / 18.0) ** 2
    src = (n1 // 2, n2 // 2, n3 // 2)
    rec = np.zeros((nt, n3, n2), np.float32)
    rec[:, 5:-5, 5:-5] = rng.standard_normal((nt, n3 - 10, n2 - 10)) * 0.1
    return c, ((1 - 2 * a) * np.exp(-a)).astype(np.float32), src, rec


def _image(hip, case, abc, j, prec):
    c, amp, src, rec = case
    g = hip.Acoustic3D(c, amp, src, min(6, c.shape[0] - 6), abc=abc, snap_every=j, snap_prec=prec)
    g.set_data(rec)
    g.migrate()
    img = g.image()
    g.close()
    return img


@pytest.mark.parametrize("prec,tol", [("fp32", 1e-4), ("bf16", 1e-2)])
@pytest.mark.parametrize("shape", [(11, 11, 11), (74, 26, 27), (75, 27, 12), (138, 31, 40), (30, 11, 160)])
def test_image_vs_fp64(hip, shape, prec, tol):
    nt, j = 60, 4
    abc = 8 if min(shape) >= 26 else 0
    print("acoustic", shape, prec, flush=True)
    case = _case(*shape, nt, 11)
    c, amp, src, rec = case
    img = _image(hip, case, abc, j, prec)
    zr = min(6, shape[0] - 6)
    _, snap = O.ac3_run(c, amp, src, zr, abc=abc, j=j, want_snap=True, nthreads=8)
    ref = O.ac3_run(c, amp, src, zr, abc=abc, mode=1, rec=rec.astype(np.float64), j=j, snap=snap, nthreads=8)
    assert np.abs(ref).max() > 0
    assert O.rel_l2(img, ref.transpose(2, 1, 0)) <= tol


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_chunking_does_not_change_results(hip, monkeypatch, prec):
    case = _case(70, 33, 47, 30, 5)
    imgs = []
    for planes in (None, "1", "7", "64"):
        if planes:
            monkeypatch.setenv("RTM_AC3_YCHUNK", planes)
        imgs.append(_image(hip, case, 8, 5, prec))
    for i in imgs[1:]:
        assert np.array_equal(i, imgs[0])
