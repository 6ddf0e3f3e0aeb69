"""The Laplace field entry under HIP graph capture as a process's first call
of it: its table of factors is built on the side, the graph holds the field
kernel alone, and replays add the same field every time."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a process of its own: the table is built once in a process
PROGRAM = r"""
import ctypes, sys
import numpy as np
import wbfmm_amd as wb
vp, sz, u, i, d = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_uint, ctypes.c_int, ctypes.c_double
L = wb.lib()
rng = np.random.default_rng(1)
n, m, N = 70, 33, 4
src, xt = rng.uniform(0.1, 0.9, (n, 3)), rng.uniform(0.1, 0.9, (m, 3))
q = rng.normal(size=n)
rows = lambda a: wb.DeviceBuffer.from_array(np.hstack([a, np.zeros((len(a), 1))]))
dev = wb.DeviceBuffer.from_array
# one box: all sources in its near field, no far field
bufs = [rows(xt), dev(np.arange(m, dtype=np.uint32)), dev(np.zeros(1, np.uint32)),
        dev(np.array([n], np.uint32)), rows(src), dev(q), dev(np.zeros((N + 1) ** 2)),
        dev(np.zeros((m, 4)))]
x0 = np.zeros(3)
s, g, ex, nodes = vp(), vp(), vp(), sz()
assert L.wbfmm_hip_stream_create(ctypes.byref(s)) == 0
wb.sync()
hip = ctypes.CDLL(next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l))
L.wbfmm_hip_set_stream(s, None)
assert hip.hipStreamBeginCapture(s, 0) == 0
xd, idd, st, en, sd, qd, md, fd = (vp(b.ptr) for b in bufs)
rc = L.wbfmm_hip_lap_field(xd, idd, u(m), st, en, sd, qd, None, None, u(0), vp(x0.ctypes.data),
                           d(1.0), i(N), md, i(3), fd, i(4))
e = hip.hipStreamEndCapture(s, ctypes.byref(g))
assert rc == 0 and e == 0, (rc, e, L.wbfmm_hip_last_error())
assert hip.hipGraphGetNodes(g, None, ctypes.byref(nodes)) == 0 and nodes.value == 1, nodes.value
assert hip.hipGraphInstantiate(ctypes.byref(ex), g, None, None, sz(0)) == 0
r = xt[:, None] - src[None]
ir = 1.0 / np.sqrt((r * r).sum(2))
want = np.hstack([(ir @ q)[:, None], -np.einsum("ts,tsc->tc", ir ** 3 * q, r)]) / (4 * np.pi)
for rep in range(4):
    bufs[7].zero()                       # eager, on the graph's stream
    assert hip.hipGraphLaunch(ex, s) == 0
    if rep % 2:
        wb.sync()
    got = bufs[7].download(np.zeros((m, 4)))
    # 70 pairs at rounding level, of the largest value of each column
    assert (np.abs(got - want).max(0) < 1e-13 * np.abs(want).max(0)).all(), rep
wb.sync()
assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(g) == 0
print("captured")
"""


def test_first_field_call_of_a_process_captured():
    r = subprocess.run([sys.executable, "-u", "-c", PROGRAM], cwd=ROOT, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "captured" in r.stdout, r.stdout + r.stderr
