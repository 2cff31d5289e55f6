"""On unstructured meshes the host chooses between two builds of RK4 (FP64) and
of AB2 / AB3 (the reduced precisions) by the elements that a step crosses.
Both sides of each choice give the same bits: FP64 against the oracle, the
Adams-Bashforth builds against the straight walks that exposure times take,
batches and served requests against particles advected frame by frame."""
import ctypes
import os
import sys

import numpy as np
import pytest

import cases
from fvcpy import fvc, host

sys.path.insert(0, os.path.join(cases.REPO, "oracle"))
import oracle  # noqa: E402
from test_gpu_element_rows import _field  # noqa: E402

pytestmark = pytest.mark.gpu

# elements of 0.2 at speeds about 1.2 (3-D): 0.02, 0.2, 0.3 and 2 elements a step
DT = [0.0033, 0.033, 0.05, 0.33]
T = 0.66


def _context(dims, precision, sl, bounds, xyz, conn, adj, nslices=2):
    ctx = fvc.Context(dims, bounds, precision, nslices, coords=xyz, conn=conn, adj=adj)
    for s in range(nslices):
        ctx.load_slice(s, T * s, sl[s % 2])
    return ctx


@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("dt", DT)
def test_f64_rk4_is_the_oracles_on_both_sides(dims, dt):
    bounds, xyz, conn, adj, sl, seeds = _field(dims)
    ctx = _context(dims, "f64", sl, bounds, xyz, conn, adj)
    om = oracle.Mesh(dims, bounds, coords=xyz, conn=conn, adj=adj)
    for s in range(2):
        om.set_slot(s, sl[s])
    om.set_interval(0.0, T)
    L = fvc.lib()
    d, i64, i32, vp = ctypes.c_double, ctypes.c_int64, ctypes.c_int32, ctypes.c_void_p
    L.fvc_advect_times.argtypes = [vp, vp, i64, i64, vp, i32, i32, d, d, vp]
    for n in (1, 65, 3000):
        recs = ctx.seed_list(seeds(n))
        for t1, t2 in ((0.0, T), (T, 0.0)):
            ref = recs.copy()
            assert om.advect(ref, t1, t2, dt) == 0
            p = fvc.Particles(ctx, n)
            p.set(recs)
            print("crossings dims %d dt %g n %d" % (dims, dt, n), flush=True)
            p.advect(t1, t2, 0, 1, 0.0, T, dt)
            got = [p.get()]
            if t2 > t1:  # the same segment for each particle
                p.set(recs)
                tt = np.tile([t1, t2], (n, 1))
                ip = fvc.IntParams(fvc.INT_RK4, 0, dt, 0, 0, 0, 0, 0.0, 0.0, 0.0)
                assert L.fvc_advect_times(ctx.h, p.h, 0, n, tt.ctypes.data_as(vp), 0, 1, 0.0, T, ctypes.byref(ip)) == 0
                got.append(p.get())
            p.close()
            for g in got:
                for k in ("X", "LeftDomain", "LeftDomainTime"):
                    np.testing.assert_array_equal(g[k], ref[k])
    ctx.close()


@pytest.mark.parametrize("precision", ["f32", "f16"])
@pytest.mark.parametrize("integrator", [fvc.INT_AB2, fvc.INT_AB3])
@pytest.mark.parametrize("dt,steps,n", [(0.0033, 12, 3000), (0.0033, 8, 3000), (0.033, 12, 3000), (0.033, 6, 70001),
                                        (0.1, 4, 70001)])
def test_adams_bashforth_is_the_straight_walks_on_both_sides(precision, integrator, dt, steps, n):
    bounds, xyz, conn, adj, sl, seeds = _field(3)
    ctx = _context(3, precision, sl, bounds, xyz, conn, adj)
    recs = ctx.seed_list(seeds(n))
    L = fvc.lib()
    L.fvc_cet_reset.argtypes = [ctypes.c_void_p]
    assert L.fvc_cet_reset(ctx.h) == 0
    out = []
    for substeps in (0, 2):
        p = fvc.Particles(ctx, n)
        p.set(recs)
        print("ab crossings %s dt %g n %d substeps %d" % (precision, dt, n, substeps), flush=True)
        ip = fvc.IntParams(integrator, 0, dt, 0, 0, 0, substeps, 0.0, 0.0, 0.0)
        assert L.fvc_advect(ctx.h, p.h, 0, n, 0.0, (steps - 0.4) * dt, 0, 1, 0.0, T, ctypes.byref(ip)) == 0
        out.append(p.get())
        p.close()
    a, b = out
    stay = a["LeftDomain"] == 0
    assert stay.sum() > n // 3
    np.testing.assert_array_equal(a["LeftDomain"], b["LeftDomain"])
    np.testing.assert_array_equal(a["X"][stay], b["X"][stay])
    np.testing.assert_array_equal(a["ElementIndex"][stay], b["ElementIndex"][stay])
    ctx.close()


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_batches_and_served_requests_on_both_sides(precision, dt):
    bounds, xyz, conn, adj, sl, seeds = _field(3)
    ctx = _context(3, precision, sl, bounds, xyz, conn, adj, 3)
    n = 1500
    recs = ctx.seed_list(seeds(2 * n))
    ref = []
    for half, it in ((0, fvc.INT_RK4), (1, fvc.INT_AB3)):
        p = fvc.Particles(ctx, n)
        p.set(recs[half * n:half * n + n])
        for f in range(2):
            p.advect(f * T, f * T + T, f, f + 1, f * T, f * T + T, dt, it)
        ref.append(p.get())
        p.close()
    ref = np.concatenate(ref)
    p = fvc.Particles(ctx, 2 * n)
    p.set(recs)
    b = fvc.Batch(ctx, p, [(0, n, 0.0, 2 * T, fvc.INT_RK4), (n, n, 0.0, 2 * T, fvc.INT_AB3)], 0.0, T, 3, dt)
    print("batch crossings %s dt %g" % (precision, dt), flush=True)
    for graph in (1, 0):
        p.set(recs)
        b.reset()
        b.run(steps_per_launch=7, use_graph=graph)
        got = p.get()
        for k in ("X", "LeftDomain", "LeftDomainTime"):
            np.testing.assert_array_equal(got[k], ref[k])
    b.close()
    s = fvc.Server(ctx, 0.0, T, 3, dt, pool_particles=100000)
    rid = s.submit_tracer(recs["X"][:n], 0.0, 2 * T)
    rif = s.submit_ftle([-0.9, -0.9, 0.5], [0.9, 0.9, 9.0], [7, 8, 20], 0.0, 2 * T)
    s.run_until_idle()
    got = s.take(rid)
    for k in ("X", "LeftDomain"):
        np.testing.assert_array_equal(got[k], ref[k][:n])
    f = fvc.FtleSlide(ctx, [-0.9, -0.9, 0.5], [0.9, 0.9, 9.0], [7, 8, 20], 1, 0.0, 2 * T)
    for k in range(2):
        f.frame(1, k, k + 1, k * T, k * T + T, dt)
    for a, w in zip(f.output(2 * T), s.take(rif)):
        np.testing.assert_array_equal(a, w)
    ctx.close()
