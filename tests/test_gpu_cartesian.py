"""RK4 on Cartesian grids against the FP64 oracle: bit for bit in FP64, over
2-D fields with and without a third component, infinite velocities, cells too
small for the shared-divisor quotients, grid nodes and walls; the reduced
precisions within a derived bound."""
import os
import sys

import numpy as np
import pytest

import cases
from fvcpy import fvc

sys.path.insert(0, os.path.join(cases.REPO, "oracle"))
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu


def _grid(dims, res, size):
    ax = [np.linspace(0.0, 1.0, r) for r in res]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    sl = []
    for s in range(2):
        u = np.stack([0.7 * np.sin(5 * y + s) + 0.3, 0.8 * np.cos(4 * x - s), 0.6 * np.sin(3 * x + 4 * z) - 0.1 * s], axis=-1)
        if dims == 2:
            u[..., 2] = 0.0
        sl.append(np.ascontiguousarray(u.reshape(-1, 3)) * size)
    return sl


def _points(dims, res, size, n, seed):
    """Points inside, on nodes and on the walls."""
    rng = np.random.default_rng(seed)
    p = rng.uniform(0.0, 1.0, (n, 3))
    k = n // 4
    p[:k] = np.round(p[:k] * (np.array(res) - 1)) / np.maximum(np.array(res) - 1, 1)
    p[:k // 4, 0] = 1.0
    if dims == 2:
        p[:, 2] = 0.0
    recs = np.zeros(n, oracle.POINT_DTYPE)
    recs["X"] = p * size
    return recs


def _both(dims, res, size, sl, recs, precision, dt, t1, t2):
    top = [size, size, size if dims == 3 else 0.0]
    b = [0.0, top[0], 0.0, top[1], 0.0, top[2]]
    kw = dict(cart_min=[0.0] * 3, cart_max=top, cart_res=res)
    ctx, om = fvc.Context(dims, b, precision, 2, **kw), oracle.Mesh(dims, b, **kw)
    for s in range(2):
        ctx.load_slice(s, float(s), sl[s])
        om.set_slot(s, sl[s])
    om.set_interval(0.0, 1.0)
    ref = recs.copy()
    assert om.advect(ref, t1, t2, dt) == 0
    p = fvc.Particles(ctx, recs.size)
    p.set(recs)
    print("cartesian dims %d res %s %s n %d" % (dims, res, precision, recs.size), flush=True)
    p.advect(t1, t2, 0, 1, 0.0, 1.0, dt)
    got = p.get()
    ctx.close()
    return got, ref


@pytest.mark.parametrize("dims,res", [(2, [2, 2, 1]), (2, [37, 18, 1]), (3, [2, 3, 2]), (3, [19, 14, 23])])
@pytest.mark.parametrize("what", ["plain", "third", "infinite", "tiny"])
@pytest.mark.parametrize("n", [1, 65, 3000])
def test_f64_bit_exact(dims, res, what, n):
    size = 1e-99 if what == "tiny" else 1.0
    sl = _grid(dims, res, size)
    if what == "third":
        sl[1][:, 2] += 0.25 * size * np.cos(np.arange(sl[1].shape[0]))
    if what == "infinite":
        sl[0][sl[0].shape[0] // 2, 0] = np.inf
        sl[1][sl[1].shape[0] // 3, 1] = -np.inf
    recs = _points(dims, res, size, n, 3)
    for t1, t2 in ((0.0, 0.31), (1.0, 0.76)):
        got, ref = _both(dims, res, size, sl, recs, "f64", 0.01, t1, t2)
        # an infinity makes the same points infinite or not a number; what becomes of those differs (the C
        # conversion of a NaN to an integer is the host's own)
        fin = np.isfinite(ref["X"]).all(axis=1)
        np.testing.assert_array_equal(np.isfinite(got["X"]).all(axis=1), fin)
        for k in ("X", "LeftDomain", "LeftDomainTime"):
            np.testing.assert_array_equal(got[k][fin], ref[k][fin])


@pytest.mark.parametrize("dims,res", [(2, [37, 18, 1]), (3, [19, 14, 23])])
@pytest.mark.parametrize("precision", ["f64", "f32", "bf16", "f16"])
def test_points_too_far_for_a_finite_quotient_are_outside(dims, res, precision):
    """(X - min) / del overflows for these points on cells of 1e-92"""
    size = 1e-90
    recs = _points(dims, res, size, 300, 8)
    recs["X"][:40, 0] = np.resize([1e250, -1e250, 1e279, -1e270, 1e300, -1e308, np.inf, -np.inf], 40)
    recs["X"][40:80, 1] = np.resize([1e250, -1e250, 1e279, -1e270, 1e300, -1e308, np.inf, -np.inf], 40)
    got, ref = _both(dims, res, size, _grid(dims, res, size), recs, precision, 0.01, 0.0, 0.05)
    assert (ref["LeftDomain"][:80] != 0).all()
    for k in ("X", "LeftDomain", "LeftDomainTime"):
        np.testing.assert_array_equal(got[k][:80], ref[k][:80])


# Against FP64: a stage velocity's relative rounding (20 roundings in FP32,
# half an ulp of the largest value in 16 bits) over T = 0.31 with |u| < 1.1 and
# gradients up to G = 5, and the FP32 local coordinates' 2^-24.
REL = {"f32": 20 * 2.0**-24, "bf16": 2.0**-9, "f16": 2.0**-12}


def _steady(dims, res, sl, recs, ref, dt, t1, t2, by):
    """Points whose FP64 exit does not change when they start `by` further
    along any axis (inwards from where that would leave the grid): none of
    their walls is so near that an error of that size could decide it."""
    same = np.ones(recs.size, bool)
    om = oracle.Mesh(dims, [0.0, 1.0, 0.0, 1.0, 0.0, 1.0 if dims == 3 else 0.0], cart_min=[0.0] * 3,
                     cart_max=[1.0, 1.0, 1.0 if dims == 3 else 0.0], cart_res=res)
    for s in range(2):
        om.set_slot(s, sl[s])
    om.set_interval(0.0, 1.0)
    for a in range(dims):
        for d in (by, -by):
            r = recs.copy()
            x = r["X"][:, a] + d
            r["X"][:, a] = np.where((x < 0.0) | (x > 1.0), r["X"][:, a] - d, x)
            assert om.advect(r, t1, t2, dt) == 0
            same &= (r["LeftDomain"] == ref["LeftDomain"]) & (np.abs(r["LeftDomainTime"] - ref["LeftDomainTime"]) < 1.5 * dt)
    return same


@pytest.mark.parametrize("dims,res", [(2, [2, 2, 1]), (2, [37, 18, 1]), (3, [2, 3, 2]), (3, [19, 14, 23])])
@pytest.mark.parametrize("precision", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("n", [1, 65, 3000])
def test_reduced_precision_follows_the_oracle(dims, res, precision, n):
    recs = _points(dims, res, 1.0, n, 5)
    sl = _grid(dims, res, 1.0)
    got, ref = _both(dims, res, 1.0, sl, recs, precision, 0.01, 0.0, 0.31)
    tol = REL[precision] * 1.1 * 0.31 * np.exp(5 * 0.31)
    stay = (got["LeftDomain"] == 0) & (ref["LeftDomain"] == 0)
    assert np.abs(got["X"][stay] - ref["X"][stay]).max(initial=0.0) <= tol
    # an exit may differ where a point comes within tol of a wall (or starts on one)
    assert (got["LeftDomain"] != ref["LeftDomain"]).sum() <= 1 + n * (0.1 + tol / 0.05)
    # and nowhere else: the points on the wall x = 1 and on the nodes among them
    sure = _steady(dims, res, sl, recs, ref, 0.01, 0.0, 0.31, 2 * tol)
    np.testing.assert_array_equal(got["LeftDomain"][sure], ref["LeftDomain"][sure])
    out = sure & (ref["LeftDomain"] != 0)
    assert np.abs(got["LeftDomainTime"][out] - ref["LeftDomainTime"][out]).max(initial=0.0) < 1.5 * 0.01
    if n == 3000:
        wall = recs["X"][:, 0] == 1.0
        assert sure.mean() > 0.5 and (sure & wall).sum() > 20 and (sure & stay).sum() > 500 and out.sum() > 100
