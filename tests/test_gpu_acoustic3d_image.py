"""Images of 3D acoustic handles read back: rows of every padding, in one piece
and in pieces by several threads, and while another thread migrates on the same
handle, which neither sees nor disturbs the run."""
import ctypes as C
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


def _free(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


# rows that a padded layout would lengthen most, and one that it lengthens by a quarter
@pytest.mark.parametrize("n1", [11, 38, 41, 66, 102])
def test_padding_takes_little_memory(hip, n1):
    """A handle takes at most a third more device memory than contiguous rows
    would (and what the allocator rounds up)."""
    n2, n3, nt, j = 150, 160, 40, 1
    rows = n2 * n3
    # velocity term, two fields, image and a snapshot a level; the record
    contiguous = 4 * n1 * rows * (4 + nt // j) + 4 * nt * rows
    warm = _handle(hip, (40, 40, 40), 3)
    warm.migrate()
    free0 = _free(hip)
    g = hip.Acoustic3D(np.full((n1, n2, n3), 0.08, np.float32, order="F"), np.ones(nt, np.float32), (5, 70, 80), 5, abc=0,
                       snap_every=j, snap_prec="fp32")
    used = free0 - _free(hip)
    print("acoustic memory", n1, used / contiguous, flush=True)
    assert used <= contiguous * 4 / 3 + 2**26
    g.close()
    warm.close()
