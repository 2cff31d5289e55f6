"""The work this framework is used for, as measurable cases.

Every case runs through the public Python entry points (fvcpy.fvc): tracers
and FTLE slides advected frame by frame between output times, batched
releases, request serving, point location and seeding.  The meshes and fields
are the repository's own generators' (pulsatile pipe, Y-bifurcation, double
gyre) and an analytic field on a 3-D Cartesian box.

listed() names the cases, draw(rng) gives one more of the same ranges,
prepare(case, seed) builds what a program holds before the call, run(state)
makes one pass, work(case) states what a pass cannot do without, and
exact(case, seed) computes a pass's outputs in 64-bit torch arithmetic.
"""
import functools
import math
import os
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "flowvc-1_amd"))

from fvcpy import fvc, host  # noqa: E402

_INT = {"euler": fvc.INT_EULER, "rk4": fvc.INT_RK4, "ab2": fvc.INT_AB2, "ab3": fvc.INT_AB3}
_MODE = {"walk": fvc.LOCATE_WALK, "global": fvc.LOCATE_GLOBAL, "walk_global": fvc.LOCATE_WALK_GLOBAL}
_TINY = 1.0e-10


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # a handful of points followed through a 2-D grid field, as in an
        # interactive look at a flow: latency and launches are all there is
        dict(name="gyre_tracers_f64", kind="tracers", field="gyre", nx=256, ny=128, precision="f64", integrator="rk4",
             n=1500, frames=2, frame_dt=0.5, dt=0.01, order="random", output="records"),
        # the plain 2-D FTLE slide of the double gyre, forward over one period
        dict(name="gyre_ftle_f64", kind="ftle", field="gyre", nx=256, ny=128, precision="f64", g0=512, g1=256, g2=1,
             frames=20, frame_dt=0.5, dt=0.01, direction=1),
        # tracers in a 3-D structured-grid field
        dict(name="box_tracers_f32", kind="tracers", field="box", nx=80, ny=64, nz=48, precision="f32", integrator="rk4",
             n=300007, frames=4, frame_dt=0.1, dt=0.005, order="random", output="xyz"),
        # a small release in a vessel: too few points to fill the chip
        dict(name="pipe_tracers_f32_small", kind="tracers", field="pipe", nx=24, nz=132, zorder=False, precision="f32",
             integrator="rk4", n=3000, frames=5, frame_dt=0.02, dt=0.001, order="random", output="xyz"),
        # the large release: renumbered mesh, tracers ordered by element,
        # positions written every tenth frame
        dict(name="pipe_tracers_f32", kind="tracers", field="pipe", nx=60, nz=330, zorder=True, precision="f32",
             integrator="rk4", n=4000000, frames=10, frame_dt=0.02, dt=0.001, order="element", output="xyz"),
        # the double-precision mode, points in the order a file lists them,
        # whole records read back
        dict(name="pipe_tracers_f64", kind="tracers", field="pipe", nx=40, nz=220, zorder=False, precision="f64",
             integrator="rk4", n=200003, frames=4, frame_dt=0.02, dt=0.001, order="random", output="records"),
        # a large 3-D FTLE slide over the whole vessel, points leaving early
        # through the wall among it
        dict(name="pipe_ftle_f32", kind="ftle", field="pipe", nx=60, nz=330, zorder=True, precision="f32", g0=96, g1=96,
             g2=480, frames=6, frame_dt=0.02, dt=0.001, direction=1),
        # a backward slide in a branching vessel from 16-bit slices
        dict(name="ybif_ftle_f16_back", kind="ftle", field="ybif", nx=92, ny=33, nz=128, zorder=False, precision="f16",
             g0=65, g1=25, g2=97, frames=5, frame_dt=0.01, dt=0.001, direction=-1),
        # uneven releases, RK4 and Adams-Bashforth mixed, in one batch
        dict(name="pipe_batch_f32", kind="batch", field="pipe", nx=40, nz=220, zorder=True, precision="f32", releases=24,
             n_lo=1000, n_hi=200000, frames=12, frame_dt=0.02, dt=0.001),
        # tracer and FTLE requests served together from 16-bit slices
        dict(name="ybif_serve_bf16", kind="serve", field="ybif", nx=92, ny=33, nz=128, zorder=False, precision="bf16",
             requests=8, n_lo=1000, n_hi=150000, frames=16, frame_dt=0.01, dt=0.001),
        # points of unknown whereabouts located in a mesh
        dict(name="pipe_locate", kind="locate", field="pipe", nx=40, nz=220, zorder=False, precision="f32", n=262147,
             mode="global"),
        # a seed list sorted for locality and located before a release
        dict(name="pipe_seeds", kind="seeds", field="pipe", nx=40, nz=220, zorder=True, precision="f32", n=1000003),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh_draw(rng):
    zorder = rng.random() < 0.5
    if rng.random() < 0.7:
        nx = rng.randint(14, 44)
        return dict(field="pipe", nx=nx, nz=int(nx * rng.uniform(4.0, 6.0)), zorder=zorder)
    nx = rng.randint(40, 110)
    return dict(field="ybif", nx=nx, ny=max(8, int(nx * 0.36)), nz=int(nx * 1.4), zorder=zorder)


def draw(rng):
    kind = rng.choice(["tracers", "tracers", "tracers", "ftle", "ftle", "batch", "serve", "locate", "seeds"])
    if kind in ("tracers", "ftle") and rng.random() < 0.35:
        if kind == "ftle" or rng.random() < 0.5:
            c = dict(field="gyre", nx=rng.randint(60, 400), ny=rng.randint(40, 200), frame_dt=0.5, dt=0.01)
        else:
            c = dict(field="box", nx=rng.randint(30, 110), ny=rng.randint(30, 90), nz=rng.randint(20, 70), frame_dt=0.1,
                     dt=0.005)
    else:
        c = _mesh_draw(rng)
        c.update(frame_dt=0.02 if c["field"] == "pipe" else 0.01, dt=0.001)
    if kind == "tracers":
        c.update(integrator=rng.choice(["rk4", "rk4", "rk4", "rk4", "ab3", "ab2", "euler"]),
                 n=_log_int(rng, 1000, 600000), frames=rng.randint(2, 8),
                 order=rng.choice(["random", "element"]) if c["field"] in ("pipe", "ybif") else "random",
                 output=rng.choice(["xyz", "records"]),
                 precision=rng.choice(["f64", "f32", "f32", "bf16", "f16"]))
    elif kind == "ftle":
        n = _log_int(rng, 4000, 400000)
        if c["field"] == "gyre":
            g1 = max(8, int(math.sqrt(n / 2)))
            c.update(g0=max(8, n // g1), g1=g1, g2=1)
        else:
            a = max(5, int((n / rng.uniform(1.5, 5.0)) ** (1.0 / 3.0)))
            c.update(g0=a, g1=max(5, a - rng.randint(0, 3)), g2=max(5, n // (a * a)))
        c.update(frames=rng.randint(2, 8), direction=rng.choice([1, -1]), precision=rng.choice(["f64", "f32", "f32", "f16"]))
    elif kind == "batch":
        c.update(releases=rng.randint(3, 32), n_lo=500, n_hi=_log_int(rng, 5000, 200000), frames=rng.randint(5, 12),
                 precision=rng.choice(["f32", "f32", "f16"]))
    elif kind == "serve":
        c.update(requests=rng.randint(2, 10), n_lo=1000, n_hi=_log_int(rng, 5000, 150000), frames=rng.randint(8, 16),
                 precision=rng.choice(["f32", "bf16", "f16"]))
    elif kind == "locate":
        c.update(n=_log_int(rng, 2000, 400000), mode=rng.choice(["global", "walk_global", "walk"]),
                 precision=rng.choice(["f64", "f32"]))
    else:
        c.update(n=_log_int(rng, 2000, 1000000), precision=rng.choice(["f64", "f32"]))
    return dict(kind=kind, **c)


# ---------------------------------------------------------------- the inputs
@functools.lru_cache(maxsize=8)
def _mesh(field, nx, ny, nz, zorder):
    """Tube, node coordinates, connectivity and adjacency; with zorder as the
    mesh renumbering writes them."""
    tube = host.pipe(nx, nx, nz, 1.0, 10.0) if field == "pipe" else host.ybif(nx, ny, nz)
    xyz, conn, adj = host.tube_mesh(tube)
    if zorder:
        _, _, xyz, conn, adj = fvc.mesh_zorder(xyz, conn, adj)
    return tube, xyz, conn, adj


def _case_mesh(c):
    return _mesh(c["field"], c["nx"], c.get("ny", c["nx"]), c["nz"], bool(c["zorder"]))


def _bounds(xyz):
    return [float(v) for a in range(3) for v in (xyz[:, a].min(), xyz[:, a].max())]


_BOX_L = (2.5, 2.0, 1.5)


def _box_slice(c, t, seed, s):
    """A swirling field on the box's nodes (x fastest), with seeded noise."""
    x, y, z = (np.linspace(0.0, L, m) for L, m in zip(_BOX_L, (c["nx"], c["ny"], c["nz"])))
    z, y, x = np.meshgrid(z, y, x, indexing="ij")
    p = 1.0 + 0.3 * math.sin(2.0 * math.pi * t)
    u = np.stack([0.8 * np.sin(2.1 * z) * p + 0.5 * np.cos(2.7 * y), 0.8 * np.sin(2.4 * x) + 0.5 * np.cos(1.9 * z) * p,
                  0.8 * np.sin(2.9 * y) + 0.5 * np.cos(2.2 * x) * p], axis=-1).reshape(-1, 3)
    return u + 0.01 * np.random.default_rng([seed, s]).standard_normal(u.shape)


def _slices(c, seed, count):
    """`count` consecutive velocity slices, one a frame."""
    fdt = c.get("frame_dt", 0.02)
    if c["field"] == "gyre":
        r = np.random.default_rng(seed)
        A, eps = 0.1 * r.uniform(0.9, 1.1), 0.25 * r.uniform(0.9, 1.1)
        return [host.double_gyre_slice(c["nx"], c["ny"], fdt * s, A, eps) for s in range(count)]
    if c["field"] == "box":
        return [_box_slice(c, fdt * s, seed, s) for s in range(count)]
    tube, xyz, _, _ = _case_mesh(c)
    with ThreadPoolExecutor(8) as ex:
        return list(ex.map(lambda s: host.tube_velocity(tube, xyz, fdt * s, 0.01, seed, s), range(count)))


def _seeds(c, n, seed):
    """n seed points in the domain, in no particular order."""
    if c["field"] == "gyre":
        r = np.random.default_rng([seed, 1])
        return np.stack([r.uniform(0.02, 1.98, n), r.uniform(0.02, 0.98, n), np.zeros(n)], axis=1)
    if c["field"] == "box":
        return np.random.default_rng([seed, 1]).uniform(0.02, 0.98, (n, 3)) * np.array(_BOX_L)
    tube = _case_mesh(c)[0]
    if c["field"] == "pipe":
        return host.tube_seeds(tube, n, 0.0, 10.0 / 3.0, seed + 1)
    return host.tube_seeds(tube, n, tube.lo[2], tube.hi[2], seed + 1)


def _nslots(c):
    return c["frames"] + 1


def _context(c, seed, slices):
    if c["field"] == "gyre":
        ctx = fvc.Context(2, [0.0, 2.0, 0.0, 1.0, 0.0, 0.0], c["precision"], max(2, len(slices)), cart_min=[0.0, 0.0, 0.0],
                          cart_max=[2.0, 1.0, 0.0], cart_res=[c["nx"], c["ny"], 1])
    elif c["field"] == "box":
        b = [v for L in _BOX_L for v in (0.0, L)]
        ctx = fvc.Context(3, b, c["precision"], max(2, len(slices)), cart_min=[0.0, 0.0, 0.0], cart_max=list(_BOX_L),
                          cart_res=[c["nx"], c["ny"], c["nz"]])
    else:
        _, xyz, conn, adj = _case_mesh(c)
        ctx = fvc.Context(3, _bounds(xyz), c["precision"], max(2, len(slices)), coords=xyz, conn=conn, adj=adj)
    for s, sl in enumerate(slices):
        ctx.load_slice(s, c["frame_dt"] * s, sl)
    return ctx


def _frames(c):
    """(tmin, tmax, lo slot, hi slot) of the frames in the order they run."""
    fdt = c["frame_dt"]
    order = range(c["frames"]) if c.get("direction", 1) > 0 else range(c["frames"] - 1, -1, -1)
    return [(f * fdt, f * fdt + fdt, f, f + 1) for f in order]


def _ftle_box(c):
    """Corners of the FTLE grid, just inside the field's bounding box."""
    if c["field"] == "gyre":
        return [0.0113, 0.0071, 0.0], [1.9891, 0.9923, 0.0]
    xyz = _case_mesh(c)[1]
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    e = hi - lo
    return (lo + e * np.array([0.0071, 0.0083, 0.0059])).tolist(), (hi - e * np.array([0.0067, 0.0079, 0.0061])).tolist()


def _ftle_times(c):
    last = _frames(c)[-1]
    return (0.0, last[1]) if c["direction"] > 0 else (_frames(c)[0][1], last[0])


def _releases(c, seed):
    r = np.random.default_rng([c["releases"], c["n_hi"]])  # how many seeds, and how moved: the case's own
    counts = np.exp(r.uniform(math.log(c["n_lo"]), math.log(c["n_hi"]), c["releases"])).astype(np.int64)
    types = r.choice([fvc.INT_RK4, fvc.INT_AB3], c["releases"])
    r = np.random.default_rng([seed, 2])
    T = c["frames"] * c["frame_dt"]
    starts = r.uniform(0.0, 0.5 * T, c["releases"])
    stops = starts + r.uniform(0.1, 1.0, c["releases"]) * (T - starts)
    out, b = [], 0
    for n, ts, te, it in zip(counts, starts, stops, types):
        out.append((b, int(n), float(ts), float(te), int(it)))
        b += int(n)
    return out


def _requests(c, seed):
    counts = np.random.default_rng([c["requests"], c["n_hi"]]).uniform(math.log(c["n_lo"]), math.log(c["n_hi"]), c["requests"])
    r = np.random.default_rng([seed, 3])
    T = c["frames"] * c["frame_dt"]
    _, xyz, _, _ = _case_mesh(c)
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    e = hi - lo
    out = []
    for q in range(c["requests"]):
        n = int(math.exp(counts[q]))
        ts = float(r.uniform(0.0, 0.5 * T))
        te = float(ts + r.uniform(0.2, 1.0) * (T - ts))
        if q % 2 == 0:
            out.append(("tracer", _seeds(c, n, seed + 17 * q), ts, te))
        else:
            h = float((e.prod() / n) ** (1.0 / 3.0))
            res = [max(4, int(round(v / h))) for v in e]
            out.append(("ftle", ((lo + 0.0071 * e).tolist(), (hi - 0.0067 * e).tolist(), res), ts, te))
    return out


def _queries(c, seed):
    """Query points over the bounding box (the corners lie outside the
    vessel) and start elements for the walks."""
    _, xyz, conn, _ = _case_mesh(c)
    r = np.random.default_rng([seed, 4])
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    if c["mode"] == "global":
        return r.uniform(lo, hi, (c["n"], 3)), None
    # points near their guesses, as a moving point's next location query
    g = r.integers(0, conn.shape[0], c["n"]).astype(np.int32)
    p = xyz[conn[g]].mean(axis=1) + r.normal(0.0, 1.0, (c["n"], 3)) * (hi - lo) / 60.0
    return p, g


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("locate", "seeds"):
        st = dict(c=c, ctx=_context(c, seed, []))
        if kind == "locate":
            st["xyz"], st["guess"] = _queries(c, seed)
        else:
            st["xyz"] = _seeds(c, c["n"], seed)
        return st
    count = max(2, c["frames"]) if kind == "serve" else _nslots(c)
    st = dict(c=c, ctx=_context(c, seed, _slices(c, seed, count)))
    ctx = st["ctx"]
    if kind == "tracers":
        recs = ctx.seed_list(_seeds(c, c["n"], seed))
        if c["order"] == "element":
            recs = _by_element(recs)
        st["ic"], st["p"] = fvc.Particles(ctx, c["n"]), fvc.Particles(ctx, c["n"])
        st["ic"].set(recs)
    elif kind == "ftle":
        mn, mx = _ftle_box(c)
        t0, t1 = _ftle_times(c)
        st["slide"] = fvc.FtleSlide(ctx, mn, mx, [c["g0"], c["g1"], c["g2"]], 1, t0, t1)
    elif kind == "batch":
        rel = _releases(c, seed)
        n = rel[-1][0] + rel[-1][1]
        st["p"] = fvc.Particles(ctx, n)
        st["p"].set(ctx.seed_list(_seeds(c, n, seed)))
        st["batch"] = fvc.Batch(ctx, st["p"], rel, 0.0, c["frame_dt"], _nslots(c), c["dt"])
    else:
        st["requests"] = _requests(c, seed)
        st["server"] = fvc.Server(ctx, 0.0, c["frame_dt"], count, c["dt"], pool_particles=4 * c["requests"] * c["n_hi"])
    return st


def _by_element(recs):
    key = np.where(recs["ElementIndex"] < 0, 1 << 30, recs["ElementIndex"])
    return recs[np.argsort(key, kind="stable")]


# ---------------------------------------------------------------- one pass
def _record_fields(recs):
    return {"x": recs["X"], "v": recs["V"], "element": recs["ElementIndex"], "left": recs["LeftDomain"],
            "left_time": recs["LeftDomainTime"]}


def run(state):
    c, ctx = state["c"], state["ctx"]
    kind = c["kind"]
    if kind == "tracers":
        p = state["p"]
        p.copy_from(state["ic"])
        p.launch_velocity(0.0, 0, 1, 0.0, c["frame_dt"])
        for tmin, tmax, lo, hi in _frames(c):
            p.advect(tmin, tmax, lo, hi, tmin, tmax, c["dt"], _INT[c["integrator"]])
        if c["output"] == "xyz":
            xyz, left = p.get_xyz()
            return {"x": xyz, "left": left}
        return _record_fields(p.get())
    if kind == "ftle":
        f = state["slide"]
        f.reset()
        for tmin, tmax, lo, hi in _frames(c):
            f.frame(c["direction"], lo, hi, tmin, tmax, c["dt"])
        t0, t1 = _ftle_times(c)
        wt, wot = f.output(abs(t1 - t0))
        return {"ftle": wt, "ftle_no_time": wot}
    if kind == "batch":
        state["batch"].reset()
        state["batch"].run()
        return _record_fields(state["p"].get())
    if kind == "serve":
        s = state["server"]
        ids = []
        for what, spec, ts, te in state["requests"]:
            ids.append(s.submit_tracer(spec, ts, te) if what == "tracer" else s.submit_ftle(*spec, ts, te))
        s.run_until_idle()
        out = []
        for (what, _, _, _), rid in zip(state["requests"], ids):
            got = s.take(rid)
            out.append(_record_fields(got) if what == "tracer" else {"ftle": got[0], "ftle_no_time": got[1]})
        return out
    if kind == "locate":
        return {"element": ctx.locate(state["xyz"], state["guess"], _MODE[c["mode"]])}
    xyz = state["xyz"]
    tube = _case_mesh(c)[0]
    perm = ctx.zsort(xyz, [tube.lo[a] for a in range(3)], [tube.hi[a] for a in range(3)])
    recs = ctx.seed_list(xyz[perm])
    return {"order": perm, "element": recs["ElementIndex"], "left": recs["LeftDomain"]}


# ---------------------------------------------------------------- its floor
def work(case):
    """Bytes: particle states in and out, and the part of the mesh and the
    slices that the pass can touch, each once.  Flops: a step's containment
    tests, interpolations and update (about 600 in a tetrahedral mesh, 250 and
    450 in a 2-D and a 3-D grid)."""
    c, kind = case, case["kind"]
    nb = {"f64": 24, "f32": 12, "bf16": 6, "f16": 6}[c["precision"]]
    if c["field"] in ("gyre", "box"):
        nodes, geom, flops = c["nx"] * c["ny"] * c.get("nz", 1), 0, 250 if c["field"] == "gyre" else 450
    else:
        vox = c["nx"] * c.get("ny", c["nx"]) * c["nz"] * (0.785 if c["field"] == "pipe" else 0.3)
        nodes, geom, flops = vox * 1.05, vox * (6 * 32 + 1.05 * 24), 600
    if kind == "locate":
        return {"bytes": c["n"] * 32.0 + min(geom, c["n"] * 300.0), "flops": c["n"] * 100.0}
    if kind == "seeds":
        return {"bytes": c["n"] * 116.0 + min(geom, c["n"] * 300.0), "flops": c["n"] * 100.0}
    per_frame = round(c["frame_dt"] / c["dt"])
    if kind == "tracers":
        n, steps = c["n"], c["n"] * c["frames"] * per_frame
        if c["integrator"] != "rk4":
            flops *= 0.4
    elif kind == "ftle":
        n = c["g0"] * c["g1"] * c["g2"]
        inside = 1.0 if c["field"] == "gyre" else 0.78 if c["field"] == "pipe" else 0.3
        steps = inside * n * c["frames"] * per_frame
    else:
        mean = (c["n_hi"] - c["n_lo"]) / math.log(c["n_hi"] / c["n_lo"])
        n = mean * c["releases" if kind == "batch" else "requests"]
        steps = n * c["frames"] * per_frame * 0.4
    touched = min(geom + nodes * nb * (c["frames"] + 1), steps * 700.0)
    return {"bytes": n * 120.0 + touched, "flops": steps * flops}


# ---------------------------------------------------------------- in 64 bits
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev()).to(dtype)


class _Mesh64:
    """Linear interpolation in a tetrahedral mesh; a position's element is
    found by walking over the adjacency from the last one."""

    def __init__(self, c, slices):
        tube, xyz, conn, adj = _case_mesh(c)
        self.adj = _t(adj, torch.int64)
        self.conn = _t(conn, torch.int64)
        X = _t(xyz)
        self.x0 = X[self.conn[:, 0]]
        a, b, d = (X[self.conn[:, q]] - self.x0 for q in (1, 2, 3))
        rows = [torch.linalg.cross(b, d), torch.linalg.cross(d, a), torch.linalg.cross(a, b)]
        self.inv = torch.stack(rows, dim=1) / (a * rows[0]).sum(dim=1).reshape(-1, 1, 1)
        self.u = [_t(s) for s in slices]
        self.lo, self.hi = X.amin(dim=0), X.amax(dim=0)
        res = [tube.nx, tube.ny, tube.nz]
        self.vlo = _t([tube.lo[a] for a in range(3)])
        self.vh = _t([(tube.hi[a] - tube.lo[a]) / res[a] for a in range(3)])
        self.res = res
        cen = sum(X[self.conn[:, q]] for q in range(4)) / 4
        v = self._voxel(cen)
        self.first = torch.full((res[0] * res[1] * res[2],), -1, dtype=torch.int64, device=X.device)
        self.first[v] = torch.arange(v.numel(), device=X.device)

    def _voxel(self, P):
        ijk = ((P - self.vlo) / self.vh).floor().to(torch.int64)
        ijk = [ijk[:, a].clamp(0, self.res[a] - 1) for a in range(3)]
        return (ijk[2] * self.res[1] + ijk[1]) * self.res[0] + ijk[0]

    def locate(self, P):
        e = self.first[self._voxel(P)]
        box = ((P < self.lo - _TINY) | (P > self.hi + _TINY)).any(dim=1)
        return self.walk(torch.where(box, -1, e), P)[0]

    def nat(self, e, P):
        rst = (self.inv[e] * (P - self.x0[e]).unsqueeze(1)).sum(dim=2)
        return torch.cat([rst, 1.0 - rst.sum(dim=1, keepdim=True)], dim=1)

    def walk(self, e, P):
        """The element holding P, -1 where the walk left the mesh (or began
        outside), and the natural coordinates there."""
        e = e.clone()
        w = torch.zeros(P.shape[0], 4, dtype=torch.float64, device=P.device)
        at = (e >= 0).nonzero().squeeze(1)
        for _ in range(100000):
            if at.numel() == 0:
                break
            ea = e[at]
            n = self.nat(ea, P[at])
            d, slot = n.min(dim=1)
            inside = d > -_TINY
            w[at[inside]] = n[inside]
            on = ~inside
            at, nxt = at[on], self.adj[ea[on], slot[on]]
            e[at] = nxt
            at = at[nxt >= 0]
        return e, w

    def velocity(self, e, P, tl, lo, hi):
        e, w = self.walk(e, P)
        k = self.conn[e.clamp(min=0)]
        w = w[:, [3, 0, 1, 2]]
        v = sum(w[:, q:q + 1] * ((1.0 - tl) * self.u[lo][k[:, q]] + tl * self.u[hi][k[:, q]]) for q in range(4))
        return torch.where((e >= 0).unsqueeze(1), v, 0.0), e

    def end(self, e, P):
        return self.walk(e, P)[0]


class _Grid64:
    """Bi- or trilinear interpolation on a Cartesian grid; a probe outside the
    grid has velocity zero and takes its point out of the domain."""

    def __init__(self, c, slices):
        self.dim = 2 if c["field"] == "gyre" else 3
        self.res = [c["nx"], c["ny"], c.get("nz", 1)]
        top = [2.0, 1.0, 0.0] if self.dim == 2 else list(_BOX_L)
        self.top = top
        self.h = [top[a] / (self.res[a] - 1) for a in range(self.dim)]
        self.u = [_t(s) for s in slices]

    def locate(self, P):
        return torch.where(self._out(P), -1, 0)

    def _out(self, P):
        bad = torch.zeros(P.shape[0], dtype=torch.bool, device=P.device)
        for a in range(3):
            bad |= (P[:, a] < -_TINY) | (P[:, a] > self.top[a] + _TINY)
        return bad

    def velocity(self, e, P, tl, lo, hi):
        bad = e < 0
        cell, loc = [], []
        for a in range(self.dim):
            q = P[:, a] / self.h[a]
            bad = bad | (q.floor() < 0) | (q.ceil() > self.res[a] - 1)
            i = q.floor().clamp(0, self.res[a] - 2)
            cell.append(i.to(torch.int64))
            loc.append(((P[:, a] - i * self.h[a]) / self.h[a]).unsqueeze(1))
        v = 0.0
        for corner in range(1 << self.dim):
            w, idx = 1.0, 0
            for a in reversed(range(self.dim)):
                b = (corner >> a) & 1
                w = w * (loc[a] if b else 1.0 - loc[a])
                idx = idx * self.res[a] + cell[a] + b
            v = v + w * ((1.0 - tl) * self.u[lo][idx] + tl * self.u[hi][idx])
        return torch.where(bad.unsqueeze(1), 0.0, v), torch.where(bad, -1, 0)

    def end(self, e, P):
        return torch.where((e < 0) | self._out(P), -1, 0)


def _advect(field, s, a, b, dt, kind, tmin, tmax, lo, hi, which=None):
    """Advances the points of s that are in the domain (of `which`, where
    given) from time a to time b between slices lo (at tmin) and hi (at tmax)."""
    live = ~s["left"] & (s["left_time"] > -_TINY)
    if which is not None:
        live &= which
    at = live.nonzero().squeeze(1)
    if at.numel() == 0:
        return
    x, e = s["x"][at], s["e"][at]
    probe = [e.clone() for _ in range(4)]
    on = torch.ones_like(e, dtype=torch.bool)
    left_time = s["left_time"][at]
    hist = s.setdefault("hist", [])
    hist = [h[at] for h in hist]
    full = math.copysign(dt, b - a)
    tc, h = a, full
    tl = lambda t: (t - tmin) / (tmax - tmin)  # noqa: E731
    while (tc - b) * (b - a) < 0.0:
        if (tc + h - b) * (tc + h - a) > 0.0:
            h = math.copysign(b - tc, b - a)
        micro = abs(h) <= 1e-12 * dt
        whole = abs(h - full) <= 1e-9 * abs(full)
        f0, p0 = field.velocity(probe[0], x, tl(tc), lo, hi)
        probe[0] = p0
        gone = p0 < 0
        order = {"ab2": 2, "ab3": 3}.get(kind, 0)
        if kind == "euler" or (order and micro):
            inc = h * f0
        elif order and whole and len(hist) >= order - 1:
            inc = h * (3 * f0 - hist[0]) / 2 if order == 2 else h * (23 * f0 - 16 * hist[0] + 5 * hist[1]) / 12
        else:
            k2, probe[1] = field.velocity(probe[1], x + 0.5 * h * f0, tl(tc + h / 2), lo, hi)
            k3, probe[2] = field.velocity(probe[2], x + 0.5 * h * k2, tl(tc + h / 2), lo, hi)
            k4, probe[3] = field.velocity(probe[3], x + h * k3, tl(tc + h), lo, hi)
            inc = h * (f0 + 2 * k2 + 2 * k3 + k4) / 6
        if kind != "euler":
            gone = (p0 < 0) | (probe[1] < 0) | (probe[2] < 0) | (probe[3] < 0)
        e1 = field.end(torch.where(on, e, -1), x + inc)
        tc = tc + h
        out = on & (gone | (e1 < 0))
        left_time = torch.where(out, tc - h, left_time)
        on = on & ~out
        x = torch.where(on.unsqueeze(1), x + inc, x)
        e = torch.where(on, e1, torch.where(out, -1, e))
        if order and not micro:
            hist = [f0] + hist[:1] if whole else []
        if order or kind == "euler":
            probe[0] = e.clone()
        probe = [torch.where(on, p, -1) for p in probe]
    s["x"][at] = x
    s["e"][at] = e
    s["left"][at] = ~on
    s["left_time"][at] = left_time
    if kind in ("ab2", "ab3"):
        keep = []
        for f in hist:
            g = torch.zeros_like(s["x"])
            g[at] = f
            keep.append(g)
        s["hist"] = keep


def _state64(field, xyz):
    x = _t(xyz).clone()
    e = field.locate(x)
    left = e < 0
    return dict(x=x, e=e, left=left, left_time=torch.where(left, -1.0, 0.0).to(torch.float64), v=torch.zeros_like(x))


def _launch(field, s, t, tmin, tmax, lo, hi):
    v, e = field.velocity(s["e"], s["x"], (t - tmin) / (tmax - tmin), lo, hi)
    s["v"] = torch.where(s["left"].unsqueeze(1), s["v"], v)
    s["left"] = s["left"] | (e < 0)


def _release64(field, c, xyz, ts, te, kind, nslots):
    """A release from ts to te over the data frames it spans."""
    s = _state64(field, xyz)
    fdt = c["frame_dt"]
    f = int(math.floor(ts / fdt))
    while f * fdt > ts:
        f -= 1
    while (f + 1) * fdt <= ts:
        f += 1
    _launch(field, s, ts, f * fdt, f * fdt + fdt, f % nslots, (f + 1) % nslots)
    while True:
        tmin = f * fdt
        tmax = tmin + fdt
        _advect(field, s, max(ts, tmin), min(te, tmax), c["dt"], kind, tmin, tmax, f % nslots, (f + 1) % nslots)
        if te - tmax < _TINY:
            return s
        f += 1


def _records64(s):
    return {"x": s["x"].cpu().numpy(), "v": s["v"].cpu().numpy(), "element": None, "left": None,
            "left_time": s["left_time"].cpu().numpy()}


def _ftle64(field, mn, mx, res, dim, t0, t1, dt, direction, frames):
    """An FTLE slide: values of points whose stencil loses a point are taken at
    the exit, the others at the end; grid index (i*res1 + j)*res2 + k."""
    dev = _dev()
    dl = [(mx[a] - mn[a]) / (res[a] - 1) if a < dim else 0.0 for a in range(3)]
    ijk = torch.meshgrid(*[torch.arange(r, device=dev) for r in res], indexing="ij")
    ijk = torch.stack([g.reshape(-1) for g in ijk], dim=1)
    x = torch.stack([mn[a] + ijk[:, a].to(torch.float64) * dl[a] for a in range(3)], dim=1)
    s = _state64(field, x.cpu().numpy())
    n = x.shape[0]
    stride = [res[1] * res[2], res[2], 1]
    everyone = torch.arange(n, device=dev)
    near, has = [], []
    for a in range(3):
        near += [everyone - stride[a], everyone + stride[a]]
        has += [ijk[:, a] > 0, ijk[:, a] < res[a] - 1]
    near = [torch.where(h, q, everyone) for q, h in zip(near, has)]
    left = s["left"]
    have = left.clone()
    for q in near:
        have |= left[q]
    wt = torch.where(left, -1.0, 0.0).to(torch.float64)
    wot = wt.clone()

    def value(pos, P, T, zero):
        """pos(axis, side) -> positions of the stencil points of P"""
        D = torch.zeros(P.numel(), 3, 3, dtype=torch.float64, device=dev)
        for a in range(dim):
            lo_edge, hi_edge = ijk[P, a] == 0, ijk[P, a] == res[a] - 1
            fac = torch.where(lo_edge | hi_edge, 1.0, 2.0).to(torch.float64)
            d = (pos(a, 1) - pos(a, 0)) / (fac * dl[a]).unsqueeze(1)
            for b in range(dim):
                D[:, b, a] = d[:, b]
        C = torch.bmm(D.transpose(1, 2).contiguous(), D)
        lam = _largest_eigenvalue(C)
        w = torch.where((lam > 1.0 - _TINY) & ~zero, 0.5 * torch.log(lam.clamp(min=1e-300)), 0.0)
        return torch.where(w == 0.0, 0.0, w / T), w

    first = True
    for tmin, tmax, lo, hi in frames:
        a = t0 if first else (tmin if direction > 0 else tmax)
        if first:
            _launch(field, s, t0, tmin, tmax, lo, hi)
            first = False
        b = min(tmax, t1) if direction > 0 else max(tmin, t1)
        before = {k: v.clone() for k, v in s.items() if k != "hist"}
        _advect(field, s, a, b, dt, "rk4", tmin, tmax, lo, hi)
        gone = s["left"] & ~before["left"]
        big = n
        trig = torch.where(gone, everyone, big)
        for q, h in zip(near, has):
            trig = torch.minimum(trig, torch.where(h & gone[q], q, big))
        P = ((trig < big) & ~have).nonzero().squeeze(1)
        if P.numel():
            te = s["left_time"][trig[P]]

            def again(Q, until):
                """Points Q from their state at the frame's start, each to its own time"""
                r = {k: before[k][Q].clone() for k in ("x", "e", "left", "left_time")}
                for stop in torch.unique(until).tolist():
                    _advect(field, r, a, stop, dt, "rk4", tmin, tmax, lo, hi, which=until == stop)
                return r

            m = P.numel()
            r = again(torch.cat([q[P] for q in near]), te.repeat(6))
            mt = te.clone()
            for k, h in enumerate(has):
                sl = slice(k * m, (k + 1) * m)
                mt = torch.minimum(mt, torch.where(h[P] & r["left"][sl], r["left_time"][sl], te))
            r = again(torch.cat([P] + [q[P] for q in near[:2 * dim]]), mt.repeat(1 + 2 * dim))
            own, nb = r["x"][:m], [r["x"][(k + 1) * m:(k + 2) * m] for k in range(2 * dim)]
            T = (mt - t0).abs()
            w1, w2 = value(lambda ax, side: torch.where(has[2 * ax + side][P].unsqueeze(1), nb[2 * ax + side], own), P,
                           T, T < _TINY)
            wt[P], wot[P] = w1, w2
            have[P] = True
    P = (~have).nonzero().squeeze(1)
    T = abs(t1 - t0)
    w1, w2 = value(lambda ax, side: s["x"][near[2 * ax + side][P]], P, T, torch.zeros_like(P, dtype=torch.bool))
    wt[P], wot[P] = w1, w2
    kji = lambda w: w.reshape(res).permute(2, 1, 0).reshape(-1).cpu().numpy()  # noqa: E731
    return {"ftle": kji(wt), "ftle_no_time": kji(wot)}


def _largest_eigenvalue(C):
    out = torch.empty(C.shape[0], dtype=torch.float64, device=C.device)
    for k in range(0, C.shape[0], 1 << 19):
        out[k:k + (1 << 19)] = torch.linalg.eigvalsh(C[k:k + (1 << 19)].cpu())[:, -1].to(C.device)
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("locate", "seeds"):  # element numbers, flags and an order: whole numbers
        return None
    count = max(2, c["frames"]) if kind == "serve" else _nslots(c)
    slices = _slices(c, seed, count)
    field = _Mesh64(c, slices) if c["field"] in ("pipe", "ybif") else _Grid64(c, slices)
    if kind == "tracers":
        xyz = _seeds(c, c["n"], seed)
        if c["order"] == "element":  # the pass's own order of these inputs
            ctx = _context(c, seed, [])
            xyz = _by_element(ctx.seed_list(xyz))["X"]
            ctx.close()
        s = _state64(field, xyz)
        fr = _frames(c)
        _launch(field, s, 0.0, 0.0, c["frame_dt"], 0, 1)
        for tmin, tmax, lo, hi in fr:
            _advect(field, s, tmin, tmax, c["dt"], c["integrator"], tmin, tmax, lo, hi)
        if c["output"] == "xyz":
            return {"x": s["x"].cpu().numpy(), "left": None}
        return _records64(s)
    if kind == "ftle":
        mn, mx = _ftle_box(c)
        t0, t1 = _ftle_times(c)
        return _ftle64(field, mn, mx, [c["g0"], c["g1"], c["g2"]], 2 if c["field"] == "gyre" else 3, t0, t1, c["dt"],
                       c["direction"], _frames(c))
    if kind == "batch":
        rel = _releases(c, seed)
        xyz = _seeds(c, rel[-1][0] + rel[-1][1], seed)
        parts = [_records64(_release64(field, c, xyz[b:b + n], ts, te, "rk4" if it == fvc.INT_RK4 else "ab3", count))
                 for b, n, ts, te, it in rel]
        return {k: None if parts[0][k] is None else np.concatenate([p[k] for p in parts]) for k in parts[0]}
    out = []
    for what, spec, ts, te in _requests(c, seed):
        if what == "tracer":
            out.append(_records64(_release64(field, c, spec, ts, te, "rk4", count)))
            continue
        fdt = c["frame_dt"]
        f = int(math.floor(ts / fdt))
        while f * fdt > ts:
            f -= 1
        while (f + 1) * fdt <= ts:
            f += 1
        fr = []
        while True:
            fr.append((f * fdt, f * fdt + fdt, f % count, (f + 1) % count))
            if te - fr[-1][1] < _TINY:
                break
            f += 1
        out.append(_ftle64(field, spec[0], spec[1], spec[2], 3, ts, te, c["dt"], 1, fr))
    return out
