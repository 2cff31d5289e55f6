"""Outputs where pinned host memory cannot be had: the same bytes as with it.
A process of its own loads a stand-in for hipHostMalloc that refuses blocks
over 256 KB before the library, and prints a digest of every kind of output."""
import os
import subprocess
import sys

import pytest

import cases

pytestmark = pytest.mark.gpu

SCRIPT = """
import ctypes, hashlib, sys
if sys.argv[1] != "-":
    ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from fvcpy import fvc, host
t = host.pipe(10, 10, 40, 1.0, 10.0)
xyz, conn, adj = host.tube_mesh(t)
ctx = fvc.Context(3, [-1.0, 1.0, -1.0, 1.0, 0.0, 10.0], "f64", 2, coords=xyz, conn=conn, adj=adj)
for s in range(2):
    ctx.load_slice(s, 0.1 * s, host.tube_velocity(t, xyz, 0.1 * s, 0.01, 3, s))
def show(what, *arrays):
    print(what, *[hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest() for a in arrays], flush=True)
for n in (7, 2000, 60000, 300001):
    x = host.tube_seeds(t, n, 0.0, 10.0, 5)
    recs = ctx.seed_list(x)
    show("seeds %d" % n, recs)
    p = fvc.Particles(ctx, n)
    p.set(recs)
    p.advect(0.0, 0.1, 0, 1, 0.0, 0.1, 0.05)
    show("records", p.get())
    show("positions", *p.get_xyz())
    show("elements", ctx.locate(x, None, fvc.LOCATE_GLOBAL))
    p.close()
show("grid", ctx.seed_grid([-0.9, -0.9, 0.5], [0.1, 0.1, 0.1], [19, 19, 90]))
for res in ([5, 6, 7], [40, 40, 200]):
    f = fvc.FtleSlide(ctx, [-0.9, -0.9, 0.5], [0.9, 0.9, 9.0], res, 1, 0.0, 0.1)
    f.frame(1, 0, 1, 0.0, 0.1, 0.05)
    show("ftle", *f.output(0.1))
    show("ftle records", f.records())
"""


def _run(shim):
    env = dict(os.environ, PYTHONPATH=os.path.join(cases.REPO, "flowvc-1_amd"))
    r = subprocess.run([sys.executable, "-c", SCRIPT, shim], capture_output=True, text=True, env=env, timeout=100)
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]
    return r.stdout


def test_outputs_without_pinned_memory_are_the_same_bytes(tmp_path):
    shim = str(tmp_path / "no_pinned.so")
    src = os.path.join(cases.REPO, "tests", "native", "no_pinned.c")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", src, "-o", shim, "-L/opt/rocm/lib", "-lamdhip64", "-ldl"], check=True)
    with_pinned = _run("-")
    print(with_pinned, flush=True)
    assert with_pinned.count("\n") == 4 * 4 + 1 + 4
    assert _run(shim) == with_pinned
