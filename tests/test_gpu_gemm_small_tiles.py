"""The small product tiles (32x32 staged 16 and 8 deep, 64x64) against the 128x64
kernel, bit for bit, at sizes on and beside their edges, every op pair,
both product forms, with and without an addend; and every one against
numpy at the same sizes.  QT_GEMM_TILE is read once per process, hence one
child process per kernel."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import sys
import numpy as np
sys.path.insert(0, sys.argv[2])
from quantum_transport_amd import rgf
rgf.init(0)
rng = np.random.default_rng(6)
cr = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
op = lambda X, o: X if o == 0 else np.swapaxes(X, 1, 2) if o == 1 else np.swapaxes(X, 1, 2).conj()
out = {}
for b, m, n, k in [(9, 1, 1, 1), (3, 31, 33, 15), (8, 32, 32, 16), (5, 33, 31, 17), (2, 64, 64, 64), (7, 65, 96, 40),
                   (3, 160, 130, 100), (2, 250, 250, 250)]:
    for oa, ob in [(0, 0), (0, 2), (2, 0), (2, 2), (0, 1), (1, 0)]:
        A = cr(b, m, k) if oa == 0 else cr(b, k, m)
        B = cr(b, k, n) if ob == 0 else cr(b, n, k)
        for prec in (rgf.QT_PREC_FP64, rgf.QT_PREC_FP64_3M):
            key = f"{b}.{m}.{n}.{k}.{oa}{ob}.{prec}"
            out[key] = rgf.zgemm_batched(A, B, oa, ob, precision=prec)
            out["d" + key] = rgf.zgemm_batched(A, B, oa, ob, alpha=-1.5, beta=0.5, R=out[key], precision=prec)
            # |error| <= gamma_k |A||B| per component, three products add their sums
            bound = 16 * (k + 4) * np.finfo(float).eps * (np.abs(op(A, oa)) @ np.abs(op(B, ob)))
            assert (np.abs(out[key] - op(A, oa) @ op(B, ob)) <= bound).all(), key
np.savez(sys.argv[1], **out)
print("gemm child done", flush=True)
"""


def test_small_tiles_bit_identical(tmp_path):
    res = {}
    for name in ("128x64w8", "32x32", "32x32k8", "64x64"):
        print("gemm child", name, flush=True)
        path = tmp_path / f"{name}.npz"
        r = subprocess.run([sys.executable, "-c", CHILD, str(path), ROOT], env=dict(os.environ, QT_GEMM_TILE=name),
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        res[name] = np.load(path)
    for key in res["128x64w8"].files:
        for other in ("32x32", "32x32k8", "64x64"):
            assert np.array_equal(res["128x64w8"][key], res[other][key]), (key, other)
