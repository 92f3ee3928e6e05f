"""Images of 3D acoustic handles read back: rows of every padding, in one piece
and in pieces by several threads, and while another thread migrates on the same
handle, which neither sees nor disturbs the run."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _handle(hip, shape, nt, j=4):
    rng = np.random.default_rng(sum(shape))
    c = np.asfortranarray(rng.uniform(0.06, 0.09, shape), np.float32)
    amp = rng.standard_normal(nt).astype(np.float32)
    g = hip.Acoustic3D(c, amp, tuple(n // 2 for n in shape), shape[0] // 2, abc=0, snap_every=j)
    rec = np.zeros((nt, shape[2], shape[1]), np.float32)
    rec[:, 5:-5, 5:-5] = 0.1 * rng.standard_normal((nt, shape[2] - 10, shape[1] - 10))
    g.set_data(rec)
    return g


# fields of 16 MiB and more come back in pieces
@pytest.mark.parametrize("shape", [(12, 11, 11), (63, 40, 37), (64, 40, 37), (150, 170, 190), (128, 190, 175)])
def test_image_equals_that_of_contiguous_rows(hip, monkeypatch, shape):
    print("acoustic image", shape, flush=True)
    out = []
    for pad in ("1", "0"):
        monkeypatch.setenv("RTM_AC3_PAD", pad)
        g = _handle(hip, shape, 24)
        g.migrate()
        out.append(g.image())
        g.close()
    assert np.array_equal(*out) and np.abs(out[0]).max() > 0


def test_image_read_during_a_migration(hip):
    g = _handle(hip, (101, 60, 70), 400)
    g.migrate()
    want = g.image()
    print("acoustic image beside a migration", flush=True)
    runs = threading.Thread(target=lambda: [g.migrate() for _ in range(5)])
    runs.start()
    reads = 0
    while runs.is_alive():
        g.image()
        reads += 1
    runs.join()
    assert reads > 1
    assert np.array_equal(g.image(), want) and np.abs(want).max() > 0
    g.close()
