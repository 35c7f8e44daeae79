"""GPU test of the launch-plan autotuner: the FP32 and precision-form
searches time their candidate plans on the first call of a shape class and
record the fastest in the tuning cache; every plan gives the same bits, so
a process that tunes and one that runs the default plans (YAEL_MI355X_TUNE=0)
return identical results."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = r'''
import hashlib, sys
sys.path.insert(0, %(root)r)
import numpy as np
import yael_amd
from yael_amd import device as dev
from yael_amd.workloads import mixture
yael_amd.init()
b = mixture(5, 200000, 128, 512, 20, centres_seed=0)
q = mixture(6, 3000, 128, 512, 20, centres_seed=0)
B, Q = dev.DeviceSet(b), dev.DeviceSet(q)
h = hashlib.sha256()
for k in (1, 10, 100):
    for rep in range(2):  # first call tunes (when enabled), second uses the plan
        i, d = dev.knn_fp32(Q, B, k)
        h.update(i.tobytes()); h.update(d.tobytes())
        i, d, _ = dev.knn_bf16(Q, B, k, max(k, 8) if k <= 16 else 2 * k)
        h.update(i.tobytes()); h.update(d.tobytes())
print("DIGEST", h.hexdigest(), flush=True)
'''


def run(env):
    r = subprocess.run([sys.executable, "-c", SCRIPT % {"root": ROOT}], env=env,
                       capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stderr[-3000:]
    line = [x for x in r.stdout.splitlines() if x.startswith("DIGEST")]
    assert line, r.stdout[-2000:]
    return line[0].split()[1]


def test_tuned_plans_give_the_default_plans_bits(tmp_path):
    cache = tmp_path / "tune.txt"
    env = dict(os.environ, YAEL_MI355X_TUNE_CACHE=str(cache))
    print("tuning run", flush=True)
    tuned = run(env)
    print("default-plan run", flush=True)
    plain = run(dict(env, YAEL_MI355X_TUNE="0"))
    assert tuned == plain
    lines = cache.read_text().split("\n")
    print("\n".join(lines), flush=True)
    # shape classes with more than one distinct candidate plan were tuned
    # (the others run their only plan) and recorded with a plan index
    # (plan indices: 3 work-item targets x 4 sketch-stride scales in both
    # forms)
    rec = [x.split() for x in lines if x.strip()]
    nplans = {"f32": 12, "bf16": 12}
    assert all(len(r) == 2 and 0 <= int(r[1]) < nplans.get(r[0].split(":")[0], 12) for r in rec)
    assert sum(r[0].startswith("f32:") for r in rec) >= 2
    assert sum(r[0].startswith("bf16:") for r in rec) >= 1


ROUTES = r'''
import ctypes, sys
sys.path.insert(0, %(root)r)
import numpy as np
import yael_amd
from yael_amd import device as dev
yael_amd.init()
L = yael_amd.lib()
def search(nq, nb, d, k, weighted):
    B, Q = dev.DeviceSet.synth(nb, d, 0, 1), dev.DeviceSet.synth(nq, d, 0, 2)
    B.compute_norms(); Q.compute_norms()
    w = None
    if weighted:
        w = dev.DeviceBuffer((nb + 31) // 32 * 32 * 4)
        one = np.ones((nb + 31) // 32 * 32, np.float32)
        yael_amd.check(L.yk_memcpy_h2d(w.ptr, one.ctypes.data_as(ctypes.c_void_p), one.nbytes), "w")
    oi, od = dev.DeviceBuffer(nq * k * 4), dev.DeviceBuffer(nq * k * 4)
    yael_amd.check(L.yk_knn_f32(2, nq, nb, d, k, Q.vec.ptr, Q.dnorm.ptr, B.vec.ptr, B.fnorm.ptr,
                                w.ptr if w else None, oi.ptr, od.ptr), "knn")
    print("searched", nq, nb, d, k, weighted, flush=True)
search(3000, 200000, 128, 100, False)
search(3000, 200000, 128, 100, True)
search(8200, 180000, 272, 10, False)  # one bucket of sizes, nq nb ld^2 below
search(8200, 240000, 272, 10, False)  # and above the lists' line
'''


def test_routes_are_tuned_apart(tmp_path):
    """A plan timed for one route, or without weights, is not taken for the
    other route or a weighted search of the same bucket of sizes."""
    cache = tmp_path / "tune.txt"
    r = subprocess.run([sys.executable, "-c", ROUTES % {"root": ROOT}],
                       env=dict(os.environ, YAEL_MI355X_TUNE_CACHE=str(cache)),
                       capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stderr[-3000:]
    print(r.stdout, cache.read_text(), flush=True)
    keys = [x.split()[0] for x in cache.read_text().split("\n") if x.strip()]
    assert set(keys) == {"f32:v2:t2:k64:ld128:q11:b17", "f32:v2:t2:k64:ld128:q11:b17:w",
                         "f32:v2:t2:k16:ld272:q13:b17", "f32:v2:t2:k16:ld272:q13:b17:lists"}
