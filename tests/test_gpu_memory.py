"""Calls whose scratch cannot be had: a launch shape that nobody recorded
gives way to one that needs none, with the same bits, and a call that fails
for lack of memory leaves nothing behind for the next one.

The cap on single allocations (tests/host/alloc_cap.cpp) has to stand in
front of the runtime before the engine is loaded, so the calls run in a
process of their own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CAP = os.path.join(HERE, "host", "_build", "liballoc_cap.so")

SCRIPT = r"""
import ctypes, sys
cap = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
cap.alloc_cap_set.argtypes = [ctypes.c_size_t]
cap.alloc_cap_set.restype = None
import numpy as np, torch
from rpmplv2_amd import robots as R, rvs, workloads as W
rng = np.random.default_rng(8)
rb = R.chain(rng.uniform(0.1, 0.3, 22), radius=0.04)
sc = W._boxes(rng, 300, 0.02, 0.2, 2.0)
sc = W.Scene(sc.dim, sc.pos * np.where(np.linalg.norm(sc.pos[:, :2], axis=1) < 0.3, 3.0, 1.0)[:, None], sc.quat,
             sc.is_ground, sc.min_dist_tol)
n = 200000
q = rng.uniform(-np.pi, np.pi, (n, 22)).astype(np.float32)
qd = torch.from_numpy(q).cuda()
def outs():
    return (torch.empty(n, device="cuda"), torch.empty((n, 22), device="cuda"),
            torch.empty(n, dtype=torch.uint8, device="cuda"))
o1, o2, o3 = outs(), outs(), outs()
torch.cuda.synchronize()
def engine():
    eng = rvs.Engine(device=0)
    return eng, eng.load_robot(rb), eng.create_env(sc)
P = rvs.PREC_FP32_REFINE
eng, rid, eid = engine()
ref = eng.distance(rid, eid, q, precision=P)[:3]
eng.close()
same = lambda got: all(np.array_equal(a, b) for a, b in zip(ref, got))
# the lists of the link-major shape take 128 bytes a configuration (25.6 MB);
# without them host arrays need about 40 MB and device arrays about 4 MB
for call, limit in (("host", 48 << 20), ("device", 16 << 20), ("async", 16 << 20)):
    eng, rid, eid = engine()
    cap.alloc_cap_set(limit)
    for repeat in range(2):
        if call == "host":
            got = eng.distance(rid, eid, q, precision=P)[:3]
        elif call == "device":
            eng.distance_device(rid, eid, qd, *o1, precision=P)
            got = [x.cpu().numpy() for x in o1]
        else:
            eng.distance_async(rid, eid, qd, *o2, precision=P)
            torch.cuda.synchronize()
            got = [x.cpu().numpy() for x in o2]
        print(call, repeat, same(got), flush=True)
        assert same(got)
    cap.alloc_cap_set(2**64 - 1)
    eng.close()
# a recorded link-major shape keeps its need: refused, and the next call runs
eng, rid, eid = engine()
eng.set_tuning(rid, eid, 4, 512, 0, 5)
cap.alloc_cap_set(16 << 20)
try:
    eng.distance_device(rid, eid, qd, *o3, precision=P)
    raise SystemExit("not refused")
except rvs.RvsError as e:
    assert e.status == rvs.RVS_ENOMEM, e
small = eng.distance(rid, eid, q[:1000], precision=P)[:3]
assert all(np.array_equal(a[:1000], b) for a, b in zip(ref, small))
print("refused, then served", flush=True)
"""


def test_shapes_without_their_scratch():
    assert os.path.exists(CAP), "liballoc_cap.so is not built: run __graft_entry__.build()"
    r = subprocess.run([sys.executable, "-u", "-c", SCRIPT, CAP], capture_output=True, text=True, timeout=110, cwd=ROOT)
    print(r.stdout[-2000:], r.stderr[-4000:])
    assert r.returncode == 0
    assert r.stdout.count("True") == 6 and "refused, then served" in r.stdout
