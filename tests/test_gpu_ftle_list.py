"""An FTLE slide keeps its list of points to integrate while few of them
leave: a slide through whose frames most points leave, a few at first, against
the served request on the same grid (which lists its points anew every frame),
and a reset slide against itself."""
import numpy as np
import pytest

from fvcpy import fvc, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("res", [[5, 5, 9], [16, 15, 33]])
def test_slide_with_points_leaving_equals_the_served_request(precision, res):
    t = host.pipe(10, 10, 30, 1.0, 10.0)
    xyz, conn, adj = host.tube_mesh(t)
    frames, fdt = 12, 0.1
    ctx = fvc.Context(3, [-1.0, 1.0, -1.0, 1.0, 0.0, 10.0], precision, frames + 1, coords=xyz, conn=conn, adj=adj)
    for s in range(frames + 1):
        ctx.load_slice(s, fdt * s, host.tube_velocity(t, xyz, fdt * s, 0.01, 3, s))
    mn, mx = [-0.93, -0.91, 7.013], [0.94, 0.92, 9.31]
    f = fvc.FtleSlide(ctx, mn, mx, res, 1, 0.0, frames * fdt)
    print("ftle list %s %s" % (precision, res), flush=True)
    out, left = [], []
    for _ in range(2):
        f.reset()
        for k in range(frames):
            f.frame(1, k, k + 1, k * fdt, k * fdt + fdt, 0.01)
            left.append(int((f.records()["LeftDomain"] != 0).sum()))
        out.append(f.output(frames * fdt))
    assert left[:frames] == left[frames:] and left[0] < left[frames // 2] < left[frames - 1]
    s = fvc.Server(ctx, 0.0, fdt, frames + 1, 0.01, pool_particles=100000)
    rid = s.submit_ftle(mn, mx, res, 0.0, frames * fdt)
    s.run_until_idle()
    out.append(s.take(rid))
    for wt, wot in out[1:]:
        np.testing.assert_array_equal(wt, out[0][0])
        np.testing.assert_array_equal(wot, out[0][1])
    ctx.close()


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_extrapolation_may_change_between_frames(precision):
    """The kept list belongs to one extrapolation flag: points that left are
    on it with extrapolation and not without.  A slide that extrapolates from
    its fourth frame on: points that have left stand still before and move on
    from there, the rest are where particles advected with the same flags are."""
    t = host.pipe(10, 10, 30, 1.0, 10.0)
    xyz, conn, adj = host.tube_mesh(t)
    flags, fdt = [0, 0, 0, 1, 1, 1], 0.1
    ctx = fvc.Context(3, [-1.0, 1.0, -1.0, 1.0, 0.0, 10.0], precision, len(flags) + 1, coords=xyz, conn=conn, adj=adj)
    for s in range(len(flags) + 1):
        ctx.load_slice(s, fdt * s, host.tube_velocity(t, xyz, fdt * s, 0.01, 3, s))
    mn, mx, res = [-0.93, -0.91, 8.513], [0.94, 0.92, 9.71], [16, 15, 21]
    f = fvc.FtleSlide(ctx, mn, mx, res, 1, 0.0, len(flags) * fdt)
    before = f.records()
    p = fvc.Particles(ctx, before.size)
    p.set(before)
    p.launch_velocity(0.0, 0, 1, 0.0, fdt)
    inside = before["LeftDomain"] == 0
    moved = 0
    for k, flag in enumerate(flags):
        print("ftle extrapolation %s frame %d flag %d" % (precision, k, flag), flush=True)
        f.frame(1, k, k + 1, k * fdt, k * fdt + fdt, 0.01, extrapolate=flag)
        p.advect(k * fdt, k * fdt + fdt, k, k + 1, k * fdt, k * fdt + fdt, 0.01, fvc.INT_RK4, flag)
        r, q = f.records(), p.get()
        np.testing.assert_array_equal(r["LeftDomain"], q["LeftDomain"])
        stay = r["LeftDomain"] == 0
        np.testing.assert_array_equal(r["X"][stay], q["X"][stay])
        gone = inside & (before["LeftDomain"] != 0)
        same = (r["X"] == before["X"]).all(axis=1)
        if flag:
            moved += int((~same[gone]).sum())
        else:
            assert same[gone].all()
        before = r
    assert moved > 100 and stay.sum() > 100
    ctx.close()
