"""Choices of the autotuner read from an RTM_TUNE_CACHE file: taken where the
tuner could have made them, made again where it could not (16-bit snapshots,
whose images go by the tile width, have width 2 only). The file is read once per
process, so each batch is created in a process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CREATE = """
import numpy as np
from elastic_amd import lib
nz, nx, nt = 130, 150, 24
coefs = [np.full((nz, nx), c, np.float32, order="F") for c in (5e-8, 5e-8, 3e5, 3e5, 9e5)]
spec = dict(nz=nz, nx=nx, xs=70, zs=20, zr=20, rx0=10, nrx=100)
b = lib.Batch(nt, 10.0, 1e-3, [spec] * 3, [coefs] * 3, np.ones(nt, np.float32), snap_every=2, snap_prec="{prec}")
print("FORM", b.txr, b.tblock)
b.close()
"""


def _create(cache, prec):
    print("tuner cache", prec, flush=True)
    env = dict(os.environ, RTM_TUNE_CACHE=str(cache), PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", CREATE.format(prec=prec)], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr
    return tuple(int(v) for v in r.stdout.split("FORM")[1].split())


# code of an entry: width + 16 * form + 256 * strip width
@pytest.mark.parametrize("prec,code,taken", [("bf16", 4, False), ("fp16", 1, False), ("bf16", 17, False),
                                             ("bf16", 2, True), ("bf16", 2 + 16, True), ("fp32", 8, True)])
def test_cached_widths(hip, tmp_path, prec, code, taken):
    made = tmp_path / "made"
    _create(made, prec)
    key = made.read_text().split()[0]
    seeded = tmp_path / "seeded"
    seeded.write_text(f"{key} {code}\n")
    form = _create(seeded, prec)
    if taken:
        assert form == (code & 15, code >> 4)
        assert len(seeded.read_text().split()) == 2  # nothing was tuned
    else:
        assert form[0] == 2
        # the new choice follows in the file and is taken from then on
        assert len(seeded.read_text().split()) == 4
        assert _create(seeded, prec) == form and len(seeded.read_text().split()) == 4
