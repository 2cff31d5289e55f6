"""Outputs (fvc_particles_get, fvc_ftle_output, ...) are written by kernels
into pinned memory: up to 256 KB in one piece, larger ones in chunks through a
ring of 1 MB (8 MB for outputs over 8 MB), host threads emptying its slots
while the next chunks are written.  Whatever the path, the host must receive
the device's bytes exactly."""
import numpy as np
import pytest

from fvcpy import fvc, host

pytestmark = pytest.mark.gpu


def _records(n, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros(n, host.POINT_DTYPE)
    r["X"] = rng.standard_normal((n, 3))
    r["V"] = rng.standard_normal((n, 3)) * 1e-300  # subnormals and tiny values survive bit for bit
    r["ElementIndex"] = rng.integers(-1, 1 << 30, n)
    r["AuxElementIndex"] = rng.integers(-1, 1 << 30, n)
    r["LeftDomain"] = rng.integers(0, 2, n)
    r["LeftDomainTime"] = rng.uniform(-1.0, 1.0, n)
    r["Scalar"] = rng.standard_normal(n)
    r["X"][:5, 0] = [0.0, -0.0, np.inf, -np.inf, 5e-324]
    return r


def _same_bytes(a, b):
    return np.array_equal(a.view(np.uint8), b.view(np.uint8))


def test_particle_records_round_trip_through_staged_copies():
    """9M records, 720 MB (687 chunks through the eight slots of the large
    ring, the last one partial); then an unaligned sub-range, and a small range
    that goes in one piece."""
    n = 9_000_000
    ctx = fvc.Context(2, [0.0, 2.0, 0.0, 1.0, 0.0, 0.0], "f64", 2, cart_min=[0, 0, 0], cart_max=[2, 1, 0],
                      cart_res=[16, 8, 1])
    recs = _records(n, 11)
    P = fvc.Particles(ctx, n)
    print("round trip of %d records" % n, flush=True)
    P.set(recs)
    assert _same_bytes(P.get(), recs)
    b = 12_345
    assert _same_bytes(P.get(n - 2 * b - 7, begin=b), recs[b:n - b - 7])
    assert _same_bytes(P.get(1000, begin=777), recs[777:1777])
    P.close()
    ctx.close()


def test_large_ftle_output_equals_a_narrow_grid_of_the_same_spacing():
    """Double-gyre FTLE on a 1101 x 1001 grid (17.6 MB: the large ring) and
    on its first 101 columns as a grid of their own (1.6 MB: the small one),
    both with spacing 2^-9 so that every grid point is the same double.
    Away from the narrow grid's last column, each point has the same stencil
    in both grids, so both fields agree bit for bit there; wot = wt * T with
    T = 2 holds on both."""
    nx, ny = 256, 128
    ctx = fvc.Context(2, [0.0, 2.0, 0.0, 1.0, 0.0, 0.0], "f64", 5, cart_min=[0, 0, 0], cart_max=[2, 1, 0],
                      cart_res=[nx, ny, 1])
    for s in range(5):
        ctx.load_slice(s, 0.5 * s, host.double_gyre_slice(nx, ny, 0.5 * s))
    h = 2.0 ** -9
    out = {}
    for name, cols in (("large", 1101), ("narrow", 101)):
        print("double gyre FTLE, %d x 1001 grid" % cols, flush=True)
        F = fvc.FtleSlide(ctx, [0.0, 0.0, 0.0], [(cols - 1) * h, 1000 * h, 0.0], [cols, 1001, 1], 1, 0.0, 2.0)
        for f in range(4):
            F.frame(1, f, f + 1, 0.5 * f, 0.5 * (f + 1), 0.01)
        wt, wot = F.output(2.0)
        out[name] = (wt.reshape(1001, cols), wot.reshape(1001, cols))
        F.close()
    (Lt, Lo), (St, So) = out["large"], out["narrow"]
    np.testing.assert_array_equal(Lt[:, :100], St[:, :100])
    np.testing.assert_array_equal(Lo[:, :100], So[:, :100])
    live = Lt > 0
    assert live.sum() > 500_000
    np.testing.assert_array_equal(Lt[live] * 2.0 == Lo[live], np.ones(live.sum(), bool))
    ctx.close()


# 80-byte records: 3,273 fill the 256 KB that go out in one piece, 13,104 the
# small ring, 104,857 is the last count of the small ring, 104,960 fill the
# large one; 28-byte positions with flags: 9,353, 37,449, 299,593 and 299,648
@pytest.mark.parametrize("n", [5, 63, 3273, 3274, 9353, 9354, 13104, 13105, 37449, 52428, 52429, 104857, 104858, 104961,
                               174763, 299593, 299594, 299649, 838860, 838861, 1700001])
def test_packed_records_and_positions_at_round_edges(n):
    ctx = fvc.Context(2, [0.0, 1.0, 0.0, 1.0, 0.0, 0.0], "f64", 2, cart_min=[0.0] * 3, cart_max=[1.0, 1.0, 0.0],
                      cart_res=[4, 4, 1])
    recs = _records(n, 9)
    p, q = fvc.Particles(ctx, n + 3), fvc.Particles(ctx, n + 3)
    p.set(recs, begin=2)
    print("packed records n %d" % n, flush=True)
    assert _same_bytes(p.get(n, begin=2), recs)
    xyz, left = p.get_xyz(n, begin=2)
    np.testing.assert_array_equal(xyz, recs["X"])
    np.testing.assert_array_equal(left, recs["LeftDomain"])
    q.copy_from(p, n, begin=1, src_begin=2)
    assert _same_bytes(q.get(n, begin=1), recs)
    ctx.close()


def test_a_large_location_gives_its_memory_back():
    """32 bytes a point are held during the call; 192 MB of them afterwards
    would be missing to later slices and particle sets."""
    t = host.pipe(6, 6, 10, 1.0, 10.0)
    xyz, conn, adj = host.tube_mesh(t)
    ctx = fvc.Context(3, [-1.0, 1.0, -1.0, 1.0, 0.0, 10.0], "f32", 2, coords=xyz, conn=conn, adj=adj)
    few = host.tube_seeds(t, 1000, 0.0, 10.0, 3)
    el = ctx.locate(few, None, fvc.LOCATE_GLOBAL)
    before = ctx.memory()[1]
    n = 6_000_000
    print("locate %d points" % n, flush=True)
    got = ctx.locate(np.resize(few, (n, 3)), None, fvc.LOCATE_GLOBAL)
    np.testing.assert_array_equal(got, np.resize(el, n))
    np.testing.assert_array_equal(ctx.locate(np.resize(few, (n, 3)), got, fvc.LOCATE_WALK), got)
    assert before - ctx.memory()[1] < 64 << 20
    ctx.close()
