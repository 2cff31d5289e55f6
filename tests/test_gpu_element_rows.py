"""The RK4 state machine of the reduced-precision modes keeps each lane's
element frame and node velocities in LDS rows.  Positions, exits and elements
against the FP64 oracle at block and wave edges, with steps from a fraction of
an element to several elements long, forward and backward."""
import ctypes
import os
import sys

import numpy as np
import pytest

import cases
from fvcpy import fvc, host

sys.path.insert(0, os.path.join(cases.REPO, "oracle"))
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu


def _field(dims):
    if dims == 3:
        t = host.pipe(10, 10, 40, 1.0, 10.0)
        xyz, conn, adj = host.tube_mesh(t)
        sl = [host.tube_velocity(t, xyz, s * 0.02, 0.01, 77, s) for s in range(2)]
        return [-1.0, 1.0, -1.0, 1.0, 0.0, 10.0], xyz, conn, adj, sl, lambda n: host.tube_seeds(t, n, 0.0, 10.0, 5)
    xyz, conn, adj = cases.chan_mesh()
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    sl = [np.stack([1.0 + np.sin(5 * xyz[:, 1] + s), 0.6 * np.cos(4 * xyz[:, 0] - s), 0 * xyz[:, 0]], axis=1) for s in range(2)]
    rng = np.random.default_rng(6)
    return ([lo[0], hi[0], lo[1], hi[1], 0.0, 0.0], xyz, conn, adj, sl, lambda n: rng.uniform(lo, hi, (n, 3)) * [1, 1, 0])


# Position error against FP64 after time T: the stage velocities carry a
# relative rounding of about 40 2^-24 in FP32 and of half an ulp of the
# slice's largest value in 16 bits (2^-9, 2^-12), so |dx| <= rel umax T e^(G T)
# with umax 3.3 and velocity gradients up to G = 4; an exit may differ only
# for points that come that close to a wall.
REL = {"f32": 40 * 2.0**-24, "bf16": 2.0**-9, "f16": 2.0**-12}


@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("precision", ["f32", "bf16", "f16"])
def test_rows_follow_the_oracle(dims, precision):
    bounds, xyz, conn, adj, sl, seeds = _field(dims)
    ctx = fvc.Context(dims, bounds, precision, 2, coords=xyz, conn=conn, adj=adj)
    om = oracle.Mesh(dims, bounds, coords=xyz, conn=conn, adj=adj)
    for s in range(2):
        ctx.load_slice(s, 0.02 * s, sl[s])
        om.set_slot(s, sl[s])
    for n in (1, 63, 65, 257, 3000):
        recs = ctx.seed_list(seeds(n))
        for dt, t1, t2 in ((1e-3, 0.0, 0.02), (0.03, 0.0, 0.24), (7e-4, 0.02, 0.0)):
            lo, hi = min(t1, t2), max(t1, t2)
            om.set_interval(lo, hi)
            ref = recs.copy()
            assert om.advect(ref, t1, t2, dt) == 0
            p = fvc.Particles(ctx, n)
            p.set(recs)
            print("rows dims %d %s n %d dt %g" % (dims, precision, n, dt), flush=True)
            p.advect(t1, t2, 0, 1, lo, hi, dt)
            got = p.get()
            p.close()
            stay = (got["LeftDomain"] == 0) & (ref["LeftDomain"] == 0)
            tol = REL[precision] * 3.3 * (hi - lo) * np.exp(4 * (hi - lo))
            assert np.abs(got["X"][stay] - ref["X"][stay]).max(initial=0.0) <= tol
            differ = (got["LeftDomain"] != ref["LeftDomain"]).sum()
            assert differ <= 1 + n * tol / 0.05
            # the element held is the one that holds the position
            at = np.ascontiguousarray(got["X"][got["LeftDomain"] == 0])
            el = got["ElementIndex"][got["LeftDomain"] == 0]
            np.testing.assert_array_equal(ctx.locate(at, el, fvc.LOCATE_WALK), el)
    ctx.close()


@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("precision", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("integrator", [fvc.INT_AB2, fvc.INT_AB3])
def test_adams_bashforth_rows_give_the_straight_walks_bits(dims, precision, integrator):
    """Extrapolation takes the straight-line build, which defines the
    Adams-Bashforth steps; points that stay must have the same bits, over two
    calls (the history is carried) that end on a clipped step."""
    bounds, xyz, conn, adj, sl, seeds = _field(dims)
    ctx = fvc.Context(dims, bounds, precision, 2, coords=xyz, conn=conn, adj=adj)
    for s in range(2):
        ctx.load_slice(s, 0.1 * s, sl[s])
    for n in (1, 64, 65, 3000):
        recs = ctx.seed_list(seeds(n))
        out = []
        for extrapolate in (0, 1):
            p = fvc.Particles(ctx, n)
            p.set(recs)
            print("ab rows dims %d %s n %d extrapolate %d" % (dims, precision, n, extrapolate), flush=True)
            steps = p.advect(0.0, 0.0405, 0, 1, 0.0, 0.1, 1e-3, integrator, extrapolate)
            steps += p.advect(0.0405, 0.1, 0, 1, 0.0, 0.1, 1e-3, integrator, extrapolate)
            out.append(p.get())
            p.close()
        a, b = out
        np.testing.assert_array_equal(a["LeftDomain"], b["LeftDomain"])
        np.testing.assert_array_equal(a["LeftDomainTime"], b["LeftDomainTime"])
        stay = a["LeftDomain"] == 0
        np.testing.assert_array_equal(a["X"][stay], b["X"][stay])
        np.testing.assert_array_equal(a["ElementIndex"][stay], b["ElementIndex"][stay])
    ctx.close()


@pytest.mark.parametrize("precision", ["f64", "f32", "bf16", "f16"])
@pytest.mark.parametrize("integrator", [fvc.INT_AB2, fvc.INT_AB3])
def test_adams_bashforth_step_may_end_past_the_loaded_interval(precision, integrator):
    """A multistep step reads the field at its start only, so the last full
    step of a call may end past the loaded interval, with the bits of the
    straight walks (which exposure times take); an RK4 step, the first of a
    history, may not."""
    bounds, xyz, conn, adj, sl, seeds = _field(3)
    ctx = fvc.Context(3, bounds, precision, 2, coords=xyz, conn=conn, adj=adj)
    for s in range(2):
        ctx.load_slice(s, 0.02 * s, sl[s])
    recs = ctx.seed_list(seeds(300))
    dt = 2.0**-10  # steps end on binary fractions, the last inside at 20 dt = 0.0195
    end = 20 * dt
    assert end < 0.02 < end + dt
    L = fvc.lib()
    L.fvc_cet_reset.argtypes = [ctypes.c_void_p]

    def advect(p, t1, t2, substeps):
        ip = fvc.IntParams(integrator, 0, dt, 0, 0, 0, substeps, 0.0, 0.0, 0.0)
        return L.fvc_advect(ctx.h, p.h, 0, 300, t1, t2, 0, 1, 0.0, 0.02, ctypes.byref(ip))

    assert L.fvc_cet_reset(ctx.h) == 0
    out = []
    for substeps in (0, 2):
        p = fvc.Particles(ctx, 300)
        p.set(recs)
        print("ab past the interval %s substeps %d" % (precision, substeps), flush=True)
        assert advect(p, 0.0, end, substeps) == 0
        assert advect(p, end, end + dt, substeps) == 0
        out.append(p.get())
        p.set(recs)
        assert advect(p, end, end + dt, substeps) == -5  # FVC_E_TLOC_RANGE
        p.close()
    a, b = out
    stay = a["LeftDomain"] == 0
    assert stay.sum() > 100
    np.testing.assert_array_equal(a["LeftDomain"], b["LeftDomain"])
    np.testing.assert_array_equal(a["X"][stay], b["X"][stay])
    np.testing.assert_array_equal(a["ElementIndex"][stay], b["ElementIndex"][stay])
    ctx.close()
