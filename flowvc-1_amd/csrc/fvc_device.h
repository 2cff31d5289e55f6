/*
 * fvc_device.h - gfx950 device code of the advection path: point location,
 * interpolation and the per-particle integrators.
 *
 * One lane owns one particle for a whole time interval; its state (FP64
 * position, walk elements of the four RK4 stage probes) lives in registers.
 * Mesh geometry and velocity are random gathers (no MFMA: this is a sparse
 * stencil, not a contraction).
 *
 * Precision modes (template MODE):
 *   P_F64  : FP64 everything, expressions in the reference's order with FP
 *            contraction off, so results are bit-identical to ompVC's.
 *   P_F32  : FP32 element frames (an inverse edge matrix and origin per
 *            element) and FP32 velocity; FP64 position/time state.  Every
 *            walk decision (accept, exit face) is taken in FP32 only when it
 *            is farther than the element's guard band from its threshold;
 *            otherwise it is recomputed with the FP64 formula, so the
 *            element sequence of a walk equals the FP64 walk's for the same
 *            query point.
 *   P_BF16/P_F16 : as P_F32 with velocity stored in 16 bits times a
 *            per-slice scale.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <type_traits>

#include "fvc_div.h"
#include "fvc_root4.h"

/* waves per SIMD the hot persistent and per-interval RK4 kernels are
 * compiled for (their VGPR budget is 512 / waves, rounded to the
 * allocation granule) */
#ifndef FVC_HOT_WAVES
#define FVC_HOT_WAVES 3
#endif

namespace fvc {

constexpr double TINY = 1.0e-10; /* ompVC/macros.h:17 */

enum Mode { P_F64 = 0, P_F32 = 1, P_BF16 = 2, P_F16 = 3 };
enum Accept { ACC_SEARCH = 0, ACC_INTERP = 1 }; /* d > -TINY (mesh.c:549) / d+TINY >= 0 (velocity.c:545) */

/* device error codes (match include/fvc.h) */
enum { E_OK = 0, E_INDET = -4, E_TLOC = -5, E_ELEM = -6, E_WALK = -7, E_EIG = -8, E_LEFT = -11, E_CET = -13 };

struct DevMesh {
    int dims, mesh_type;
    double bounds[6];
    /* Cartesian velocity grid */
    double cmin[3], cdel[3];
    double cinv[3]; /* 1 / cdel rounded to nearest, 0 where div_near does not apply */
    double cfar[3]; /* twice the grid's extent: what lies as far from cmin is outside, nearer quotients are finite */
    int cres[3];
    /* unstructured */
    const double4 *__restrict__ X64;
    const float4 *__restrict__ ER; /* FP32 affine frame of each element (4 x float4) */
    const int4 *__restrict__ conn;
    const int4 *__restrict__ adj;
    double centre[3];
    int64_t nn, ne;
    float gq;       /* FP32 guard coefficient of the query offset: 12 2^-24 max |M| */
    int walk_limit; /* hop limit */
    /* spatial hash */
    const int *__restrict__ cell_start;
    const int *__restrict__ cell_elems;
    double hlo[3], hinv[3];
    int hres[3];
};

enum { VALS_INF = 1, VALS_Z = 2 }; /* an infinity; a third component other than zero */

/* Velocity slices bound for one interval: slot lo at tmin, hi at tmax. */
struct DevField {
    const void *lo, *hi;
    float scale_lo, scale_hi;
    double tmin, tmax;
    /* what the FP64 values of the two slices may hold (Cartesian meshes) */
    int vals = VALS_INF | VALS_Z;
    float crossings = 0.0f; /* for the host's choice of a build: rms speed over the mean element edge */
    /* strain-rate slices at tmin, tmax when the activation potential is integrated, else null */
    const double *sr_lo = nullptr, *sr_hi = nullptr;
    /* exposure time accumulators (per element: 128-bit fixed-point time, encounters), else null */
    unsigned long long *cet_lo = nullptr, *cet_hi = nullptr;
    int *cet_enc = nullptr;
    int cet_sub = 0; /* Trace_CETSubsteps */
    /* Runge-Kutta-Fehlberg: Int_MinTimeStep, Int_MaxTimeStep, Int_Accuracy */
    double rkf_min = 0.0, rkf_max = 0.0, rkf_tol = 0.0;
};

struct ErrBuf {
    int *code;     /* first error */
    int64_t *where;
};

__device__ inline void raise_err(ErrBuf e, int code, int64_t where) {
    if (atomicCAS(e.code, 0, code) == 0) *e.where = where;
}

/* Gather of element idx of an unstructured-mesh array with a 32-bit byte
 * offset: node, connectivity, adjacency and node-velocity arrays are below
 * 4 GiB (fvc_create checks it), so the address is the array base plus a
 * zero-extended 32-bit offset, which gfx950's global loads take as a scalar
 * base and one vector register, without 64-bit address arithmetic. */
template <typename T>
__device__ __forceinline__ T ld32(const T *__restrict__ base, uint32_t idx) {
    const uint32_t off = idx * (uint32_t)sizeof(T);
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + (uint64_t)off);
}

/* A wave claims the next 64 entries of a persistent kernel's work queue
 * (a counter per queue, reset before the launch) and returns their offset;
 * an offset >= len means the queue is exhausted.  Lane 0 reads the counter
 * first and skips the atomic once it has passed len, so the waves that
 * arrive after the queue ran out (most of a launch with little work) do not
 * all contend on one address; the counter only grows, so a stale read only
 * costs an atomic. */
__device__ __forceinline__ int claim64(int *queue, int len) {
    int base = 0;
    if ((threadIdx.x & 63) == 0) {
        base = __hip_atomic_load(queue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (base < len) base = atomicAdd(queue, 64);
    }
    return __shfl(base, 0, 64);
}

/* ------------------------------------------------------------------------ */
/* FP64 natural coordinates in the reference's expression order               */
/* (ompVC/mesh.c:527-547, velocity.c:497-517)                                */
/* ------------------------------------------------------------------------ */
__device__ __forceinline__ void nat3_exact_p(const double4 *__restrict__ X64, const int4 *__restrict__ conn, int e,
                                             double x, double y, double z, double &r, double &s, double &t) {
#pragma clang fp contract(off)
    int4 nd = ld32(conn, e);
    double4 p0 = ld32(X64, nd.x), p1 = ld32(X64, nd.y), p2 = ld32(X64, nd.z), p3 = ld32(X64, nd.w);
    double x0 = p0.x, y0 = p0.y, z0 = p0.z, x1 = p1.x, y1 = p1.y, z1 = p1.z;
    double x2 = p2.x, y2 = p2.y, z2 = p2.z, x3 = p3.x, y3 = p3.y, z3 = p3.z;
    double c11 = (z3 - z0) * (y2 - y3) - (z2 - z3) * (y3 - y0);
    double c21 = (z3 - z0) * (y0 - y1) - (z0 - z1) * (y3 - y0);
    double c31 = (z1 - z2) * (y0 - y1) - (z0 - z1) * (y1 - y2);
    double c12 = (x3 - x0) * (z2 - z3) - (x2 - x3) * (z3 - z0);
    double c22 = (x3 - x0) * (z0 - z1) - (x0 - x1) * (z3 - z0);
    double c32 = (x1 - x2) * (z0 - z1) - (x0 - x1) * (z1 - z2);
    double c13 = (y3 - y0) * (x2 - x3) - (y2 - y3) * (x3 - x0);
    double c23 = (y3 - y0) * (x0 - x1) - (y0 - y1) * (x3 - x0);
    double c33 = (y1 - y2) * (x0 - x1) - (y0 - y1) * (x1 - x2);
    double det = (x1 - x0) * ((y2 - y0) * (z3 - z0) - (z2 - z0) * (y3 - y0)) +
                 (x2 - x0) * ((y0 - y1) * (z3 - z0) - (z0 - z1) * (y3 - y0)) +
                 (x3 - x0) * ((y1 - y0) * (z2 - z0) - (z1 - z0) * (y2 - y0));
    double dx = x - x0, dy = y - y0, dz = z - z0;
    r = (c11 * dx + c12 * dy + c13 * dz) / det;
    s = (c21 * dx + c22 * dy + c23 * dz) / det;
    t = (c31 * dx + c32 * dy + c33 * dz) / det;
}

__device__ __forceinline__ void nat2_exact_p(const double4 *__restrict__ X64, const int4 *__restrict__ conn, int e,
                                             double x, double y, double &r, double &s) {
#pragma clang fp contract(off)
    int4 nd = ld32(conn, e);
    double4 p0 = ld32(X64, nd.x), p1 = ld32(X64, nd.y), p2 = ld32(X64, nd.z);
    double x0 = p0.x, y0 = p0.y, x1 = p1.x, y1 = p1.y, x2 = p2.x, y2 = p2.y;
    double c11 = y2 - y0, c12 = x0 - x2, c21 = y0 - y1, c22 = x1 - x0;
    double det = (x1 - x0) * (y2 - y0) - (x2 - x0) * (y1 - y0);
    r = (c11 * (x - x0) + c12 * (y - y0)) / det;
    s = (c21 * (x - x0) + c22 * (y - y0)) / det;
}

__device__ __forceinline__ void nat3_exact(const DevMesh &m, int e, double x, double y, double z, double &r, double &s,
                                           double &t) {
    nat3_exact_p(m.X64, m.conn, e, x, y, z, r, s, t);
}

__device__ __forceinline__ void nat2_exact(const DevMesh &m, int e, double x, double y, double &r, double &s) {
    nat2_exact_p(m.X64, m.conn, e, x, y, r, s);
}

__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }

/* exact decision on natural coordinates; returns 1 accept, 0 move (slot set), -1 indeterminate */
template <int DIM>
__device__ __forceinline__ int decide_exact(double r, double s, double t, int acc, int &slot, int *tie = nullptr) {
#pragma clang fp contract(off)
    double d, l0;
    if (DIM == 3) {
        l0 = 1 - r - s - t;
        d = dmin(r, dmin(s, dmin(t, l0)));
    } else {
        l0 = 1 - r - s;
        d = dmin(r, dmin(s, l0));
    }
    if (tie && d == -TINY) *tie = 1; /* the one value on which the two acceptance rules differ */
    bool in = acc == ACC_SEARCH ? (d > -TINY) : ((d + TINY) >= 0);
    if (in) return 1;
    if (fabs(r - d) < TINY) slot = 0;
    else if (fabs(s - d) < TINY) slot = 1;
    else if (DIM == 3 && fabs(t - d) < TINY) slot = 2;
    else if (fabs(d - l0) < TINY) slot = DIM == 3 ? 3 : 2;
    else return -1;
    return 0;
}

/* ------------------------------------------------------------------------ */
/* FP32 natural coordinates from per-element affine frames                  */
/* ------------------------------------------------------------------------ */
/* Element e's frame is four float4 at ER[4e .. 4e+3], built at fvc_create
 * from the FP64 nodes (relative to the mesh centre):
 *   ER[4e+a] = (M[a][0], M[a][1], M[a][2], o[a])   a = 0, 1, 2
 *   ER[4e+3] = (lo[0], lo[1], lo[2], g)
 * o = node 0 rounded to FP32 (an FP32 origin, exact in FP32), M = the inverse
 * of the edge matrix [n1-n0, n2-n0, n3-n0] rounded to FP32, lo the natural
 * coordinates of o itself (o - node0 is the rounding of node 0), and g the
 * element's guard coefficient 4 (18 cond + 12) 2^-24, cond = |M| |E| in the
 * row-sum norm with the 1-r-s-t row included.  2-D frames use the (x, y)
 * parts of rows 0, 1 and 3.  Natural coordinates are then
 *   (r, s, t) = lo + M (q - o),
 * q - o formed as (A - o) + d from the anchor A and offset d of the query
 * (or rounded once from the FP64 difference), three FMAs per coordinate.
 * Per coordinate, the rounding of M, of (A - o), of the sum with d and of
 * the three FMAs err by at most 6 2^-24 cond L + 2^-24 |M| |d| to first
 * order, L = max(1, |r|, |s|, |t|, |1-r-s-t|); 1-r-s-t sums three such
 * errors and rounds three times more: (18 cond + 12) 2^-24 L +
 * 3 2^-24 |M| |d| in all, and the band is four times that.  Node rounding
 * enters only through lo, so the band scales with the element's own shape,
 * not with the mesh's extent.  An element whose edge matrix is singular or
 * whose frame is not finite gets M = 0, lo = 0, g = inf: every test on it
 * is decided in FP64. */
struct Frame {
    float4 a0, a1, a2, a3;
};

template <int DIM>
__device__ __forceinline__ Frame ld_frame(const DevMesh &m, int e) {
    Frame F;
    const uint32_t b = 4u * (uint32_t)e;
    F.a0 = ld32(m.ER, b);
    F.a1 = ld32(m.ER, b + 1);
    if (DIM == 3) F.a2 = ld32(m.ER, b + 2);
    else F.a2 = make_float4(0.f, 0.f, 0.f, 0.f);
    F.a3 = ld32(m.ER, b + 3);
    return F;
}

/* (r, s, t) = lo + M q with q = query - o, each an explicit FMA chain */
template <int DIM>
__device__ __forceinline__ void frame_nat(const Frame &F, float qx, float qy, float qz, float &r, float &s, float &t) {
    if (DIM == 3) {
        r = __builtin_fmaf(F.a0.z, qz, __builtin_fmaf(F.a0.y, qy, __builtin_fmaf(F.a0.x, qx, F.a3.x)));
        s = __builtin_fmaf(F.a1.z, qz, __builtin_fmaf(F.a1.y, qy, __builtin_fmaf(F.a1.x, qx, F.a3.y)));
        t = __builtin_fmaf(F.a2.z, qz, __builtin_fmaf(F.a2.y, qy, __builtin_fmaf(F.a2.x, qx, F.a3.z)));
    } else {
        r = __builtin_fmaf(F.a0.y, qy, __builtin_fmaf(F.a0.x, qx, F.a3.x));
        s = __builtin_fmaf(F.a1.y, qy, __builtin_fmaf(F.a1.x, qx, F.a3.y));
        t = 0.0f;
    }
}

/* query given in FP64 (x, y, z): q - o rounded once from the FP64 difference */
template <int DIM>
__device__ __forceinline__ void nat_fast(const DevMesh &m, int e, double x, double y, double z, float &r, float &s,
                                         float &t, float &ge) {
#pragma clang fp contract(off)
    const Frame F = ld_frame<DIM>(m, e);
    const float qx = (float)((x - m.centre[0]) - (double)F.a0.w);
    const float qy = (float)((y - m.centre[1]) - (double)F.a1.w);
    const float qz = DIM == 3 ? (float)((z - m.centre[2]) - (double)F.a2.w) : 0.0f;
    frame_nat<DIM>(F, qx, qy, qz, r, s, t);
    ge = F.a3.w;
}

/* query anchored in FP32: the point (centre + A) + d, q - o = (A - o) + d */
template <int DIM>
__device__ __forceinline__ void nat_frame(const Frame &F, const float A[3], const float d[3], float &r, float &s,
                                          float &t, float &ge) {
#pragma clang fp contract(off)
    const float qx = (A[0] - F.a0.w) + d[0];
    const float qy = (A[1] - F.a1.w) + d[1];
    const float qz = DIM == 3 ? (A[2] - F.a2.w) + d[2] : 0.0f;
    frame_nat<DIM>(F, qx, qy, qz, r, s, t);
    ge = F.a3.w;
}

template <int DIM>
__device__ __forceinline__ void nat_fast_c(const DevMesh &m, int e, const float A[3], const float d[3], float &r,
                                           float &s, float &t, float &ge) {
    nat_frame<DIM>(ld_frame<DIM>(m, e), A, d, r, s, t, ge);
}

/* guard term of a query offset d (its rounding in (A - o) + d) */
__device__ __forceinline__ float guard_offset(const DevMesh &m, const float d[3]) {
    return m.gq * fmaxf(fabsf(d[0]), fmaxf(fabsf(d[1]), fabsf(d[2])));
}

/* FP32 decision: 1 accept, 0 move (slot set), 2 undecided (escalate); the
 * band is ge L + gq around each threshold */
template <int DIM>
__device__ __forceinline__ int decide_fast(float r, float s, float t, float ge, float gq, int &slot) {
#pragma clang fp contract(off)
    const float l0 = DIM == 3 ? ((1.0f - r) - s) - t : (1.0f - r) - s;
    /* smallest and second smallest by pairs, without arrays (a dynamically
     * indexed array would go through LDS) */
    const float lo1 = fminf(r, s), hi1 = fmaxf(r, s);
    const float lo2 = DIM == 3 ? fminf(t, l0) : l0, hi2 = DIM == 3 ? fmaxf(t, l0) : 3.0e38f;
    const float d = fminf(lo1, lo2);
    const float L = fmaxf(fmaxf(fabsf(r), fabsf(s)), DIM == 3 ? fmaxf(fabsf(t), fabsf(l0)) : fabsf(l0));
    const float g = __builtin_fmaf(ge, fmaxf(L, 1.0f), gq);
    const bool num = r == r; /* a query that is not a number moves on through slot 0 */
    if (d > g && num) return 1;
    slot = 0;
    if (!num) return 0;
    if (d >= -g) return 2;
    const float second = fminf(fmaxf(lo1, lo2), fminf(hi1, hi2));
    if (second - d <= 2.0f * g) return 2;
    if (s == d) slot = 1;
    if (DIM == 3) {
        if (t == d) slot = 2;
        if (l0 == d) slot = 3;
    } else if (l0 == d) {
        slot = 2;
    }
    return 0;
}

/* ------------------------------------------------------------------------ */
/* walk (ompVC/mesh.c:496-611 and velocity.c:523-600)                       */
/* ------------------------------------------------------------------------ */
/* Walks from `e` towards (x,y,z).  Returns the accepting element, -1 when an
 * adjacency of -1 is crossed, or -2 on error (err set).  Natural coordinates
 * of the accepting element are returned in r,s,t (for interpolation). */
template <int MODE, int DIM>
__device__ __forceinline__ int walk(const DevMesh &m, double x, double y, double z, int e, int acc, double &r, double &s,
                                    double &t, int &err, int *tie = nullptr) {
    for (int hop = 0; hop < m.walk_limit; hop++) {
        int slot = -1, dec;
        if constexpr (MODE == P_F64) {
            if (DIM == 3) nat3_exact(m, e, x, y, z, r, s, t);
            else {
                nat2_exact(m, e, x, y, r, s);
                t = 0.0;
            }
            dec = decide_exact<DIM>(r, s, t, acc, slot, tie);
        } else {
            float fr, fs, ft, ge;
            nat_fast<DIM>(m, e, x, y, z, fr, fs, ft, ge);
            dec = decide_fast<DIM>(fr, fs, ft, ge, 0.0f, slot);
            if (dec == 2) {
                if (DIM == 3) nat3_exact(m, e, x, y, z, r, s, t);
                else {
                    nat2_exact(m, e, x, y, r, s);
                    t = 0.0;
                }
                dec = decide_exact<DIM>(r, s, t, acc, slot, tie);
            } else {
                r = fr;
                s = fs;
                t = ft;
            }
        }
        if (dec == 1) return e;
        if (dec < 0) {
            err = E_INDET;
            return -2;
        }
        e = ld32(reinterpret_cast<const int *>(m.adj), 4 * (uint32_t)e + slot);
        if (e == -1) return -1;
    }
    err = E_WALK;
    return -2;
}

/* ------------------------------------------------------------------------ */
/* walk on a query point given in FP32 relative to the mesh centre           */
/* ------------------------------------------------------------------------ */
/* The RK4 stage probes of the reduced-precision modes are formed in FP32 as
 * an anchor A = (float)(X - centre) and a small offset d = D + c h k, D the
 * FP32 residual of X - centre - A; the probe stands for the point
 * (centre + A) + d.  The offset keeps FP32 resolution at its own small
 * magnitude, so probes sit within ~1e-10 of the FP64 probe positions.  An
 * FP32 decision forms q - node0 as (A - node0) + d, and an undecided one is
 * recomputed with the FP64 formula at (centre + A) + d, so the element
 * returned is the one the reference's walk returns for that point. */
/* the FP64 decision at the double point (x, y, z), for the few tests that
 * fall inside the guard band (node coordinates and connectivity by pointer,
 * so the call can stay out of line without the mesh descriptor); tie reports
 * d == -TINY, where the two acceptance rules differ */
struct ExactDec {
    float r, s, t;
    int slot, dec, tie;
};

/* inlined: an out-of-line call costs the hot kernels registers around the
 * call (build with FVC_ESC_NOINLINE to compare) */
#ifdef FVC_ESC_NOINLINE
#define FVC_ESC_ATTR __noinline__
#else
#define FVC_ESC_ATTR __forceinline__
#endif

template <int DIM>
__device__ FVC_ESC_ATTR ExactDec decide_exact_at(const double4 *__restrict__ X64, const int4 *__restrict__ conn, int e,
                                                 double x, double y, double z, int acc) {
#pragma clang fp contract(off)
    double r, s, t = 0.0;
    if (DIM == 3) nat3_exact_p(X64, conn, e, x, y, z, r, s, t);
    else nat2_exact_p(X64, conn, e, x, y, r, s);
    ExactDec o;
    o.slot = -1;
    o.tie = 0;
    o.dec = decide_exact<DIM>(r, s, t, acc, o.slot, &o.tie);
    o.r = (float)r;
    o.s = (float)s;
    o.t = (float)t;
    return o;
}

/* walk<MODE != P_F64> with the query point (centre + A) + d: returns the
 * accepting element, -1 when an adjacency of -1 is crossed, -2 on error */
template <int DIM>
__device__ __forceinline__ int walk_c(const DevMesh &m, const float A[3], const float d[3], int e, int acc, float &r,
                                      float &s, float &t, int4 &nodes, int &err) {
    const float gd = guard_offset(m, d);
    for (int hop = 0; hop < m.walk_limit; hop++) {
        int slot = -1;
        nodes = ld32(m.conn, e);
        float fr, fs, ft, ge;
        nat_fast_c<DIM>(m, e, A, d, fr, fs, ft, ge);
        int dec = decide_fast<DIM>(fr, fs, ft, ge, gd, slot);
        if (dec == 2) {
            const ExactDec x = decide_exact_at<DIM>(m.X64, m.conn, e, (m.centre[0] + (double)A[0]) + (double)d[0],
                                                    (m.centre[1] + (double)A[1]) + (double)d[1],
                                                    (m.centre[2] + (double)A[2]) + (double)d[2], acc);
            fr = x.r;
            fs = x.s;
            ft = x.t;
            slot = x.slot;
            dec = x.dec;
        }
        if (dec == 1) {
            r = fr;
            s = fs;
            t = ft;
            return e;
        }
        if (dec < 0) {
            err = E_INDET;
            return -2;
        }
        e = ld32(reinterpret_cast<const int *>(m.adj), 4 * (uint32_t)e + slot);
        if (e == -1) return -1;
    }
    err = E_WALK;
    return -2;
}

/* ------------------------------------------------------------------------ */
/* searches (ompVC/mesh.c:304-398, 496-611)                                  */
/* ------------------------------------------------------------------------ */
/* Whether element e holds (x, y, z), d > -TINY (mesh.c:321-363): by the FP32
 * frame where the smallest natural coordinate is clear of the guard band, else
 * by the FP64 formula. */
template <int DIM>
__device__ __forceinline__ bool holds(const DevMesh &m, int e, double x, double y, double z) {
    float fr, fs, ft, ge;
    nat_fast<DIM>(m, e, x, y, z, fr, fs, ft, ge);
    {
#pragma clang fp contract(off)
        const float l0 = DIM == 3 ? ((1.0f - fr) - fs) - ft : (1.0f - fr) - fs;
        float d = fminf(fminf(fr, fs), l0), L = fmaxf(fmaxf(fabsf(fr), fabsf(fs)), fabsf(l0));
        if (DIM == 3) {
            d = fminf(d, ft);
            L = fmaxf(L, fabsf(ft));
        }
        const float g = ge * fmaxf(L, 1.0f);
        if (d > g) return true;
        if (d < -g) return false;
    }
    double r, s, t = 0.0;
    if (DIM == 3) nat3_exact(m, e, x, y, z, r, s, t);
    else nat2_exact(m, e, x, y, r, s);
    int slot;
    return decide_exact<DIM>(r, s, t, ACC_SEARCH, slot) == 1;
}

/* the cell of (x, y, z) in the spatial hash, -1 outside it */
template <int DIM>
__device__ __forceinline__ int64_t hash_cell(const DevMesh &m, double x, double y, double z) {
    double fx = (x - m.hlo[0]) * m.hinv[0], fy = (y - m.hlo[1]) * m.hinv[1];
    double fz = DIM == 3 ? (z - m.hlo[2]) * m.hinv[2] : 0.0;
    if (!(fx >= 0.0 && fy >= 0.0 && fz >= 0.0)) return -1;
    if (!(fx < (double)m.hres[0] && fy < (double)m.hres[1] && fz < (double)m.hres[2])) return -1;
    return ((int64_t)(int)fz * m.hres[1] + (int)fy) * m.hres[0] + (int)fx;
}

/* lowest-index element holding the point, -1 where none does; cell lists are
 * ascending, so the first pass is the lowest index.  A cell lists some 40
 * elements: by their frames, and no further than the first that holds the
 * point, 262,147 points in 1.7M tets take 131 us, by the FP64
 * formula over whole lists (to a second holding element) 622. */
template <int DIM>
__device__ int hash_global(const DevMesh &m, double x, double y, double z) {
    const int64_t cell = hash_cell<DIM>(m, x, y, z);
    if (cell < 0) return -1;
    for (int q = m.cell_start[cell], end = m.cell_start[cell + 1]; q < end; q++) {
        const int e = m.cell_elems[q];
        if (holds<DIM>(m, e, x, y, z)) return e;
    }
    return -1;
}

/* every element with d > -TINY, ascending: the first `cap` are written to
 * `list` (when given), the lowest is returned in `first`, the count is
 * returned whole */
template <int DIM>
__device__ int hash_accepting(const DevMesh &m, double x, double y, double z, int *list, int cap, int &first) {
    first = -1;
    const int64_t cell = hash_cell<DIM>(m, x, y, z);
    if (cell < 0) return 0;
    int cnt = 0;
    for (int q = m.cell_start[cell], end = m.cell_start[cell + 1]; q < end; q++) {
        const int e = m.cell_elems[q];
        if (holds<DIM>(m, e, x, y, z)) {
            if (cnt == 0) first = e;
            if (list && cnt < cap) list[cnt] = e;
            cnt++;
        }
    }
    return cnt;
}

/* the FP64 walk's element (mesh.c:496-611) by FP32 frames where they decide;
 * a point that is not a number is left to the FP64 formula, whose comparisons
 * all fail on it */
template <int DIM>
__device__ int local_search(const DevMesh &m, double x, double y, double z, int e, int &err) {
    for (int hop = 0; hop < m.walk_limit; hop++) {
        int slot = -1;
        float fr, fs, ft, ge;
        nat_fast<DIM>(m, e, x, y, z, fr, fs, ft, ge);
        int dec = decide_fast<DIM>(fr, fs, ft, ge, 0.0f, slot);
        if (dec == 2 || fr != fr) {
            double r, s, t = 0.0;
            if (DIM == 3) nat3_exact(m, e, x, y, z, r, s, t);
            else nat2_exact(m, e, x, y, r, s);
            dec = decide_exact<DIM>(r, s, t, ACC_SEARCH, slot);
        }
        if (dec == 1) return e;
        if (dec < 0) {
            err = E_INDET;
            return -1;
        }
        e = ld32(reinterpret_cast<const int *>(m.adj), 4 * (uint32_t)e + slot);
        if (e == -1) return -1;
    }
    err = E_WALK;
    return -1;
}

/* ------------------------------------------------------------------------ */
/* velocity loads                                                            */
/* ------------------------------------------------------------------------ */
template <int MODE>
struct VelT {
    using T = double;
};
template <>
struct VelT<P_F32> {
    using T = float;
};
template <>
struct VelT<P_BF16> {
    using T = float;
};
template <>
struct VelT<P_F16> {
    using T = float;
};

/* velocity of node n of an unstructured mesh (32-bit offsets, see ld32) */
template <int MODE>
__device__ __forceinline__ void load_vel_node(const void *base, float scale, uint32_t n, typename VelT<MODE>::T out[3]) {
    if constexpr (MODE == P_F64) {
        const double4 v = ld32(reinterpret_cast<const double4 *>(base), n);
        out[0] = v.x;
        out[1] = v.y;
        out[2] = v.z;
    } else if constexpr (MODE == P_F32) {
        const float4 v = ld32(reinterpret_cast<const float4 *>(base), n);
        out[0] = v.x;
        out[1] = v.y;
        out[2] = v.z;
    } else {
        const uint2 w = ld32(reinterpret_cast<const uint2 *>(base), n);
        unsigned short h0 = (unsigned short)(w.x & 0xffffu), h1 = (unsigned short)(w.x >> 16);
        unsigned short h2 = (unsigned short)(w.y & 0xffffu);
        if constexpr (MODE == P_BF16) {
            out[0] = __uint_as_float((unsigned)h0 << 16) * scale;
            out[1] = __uint_as_float((unsigned)h1 << 16) * scale;
            out[2] = __uint_as_float((unsigned)h2 << 16) * scale;
        } else {
            out[0] = __half2float(__ushort_as_half(h0)) * scale;
            out[1] = __half2float(__ushort_as_half(h1)) * scale;
            out[2] = __half2float(__ushort_as_half(h2)) * scale;
        }
    }
}

template <int MODE>
__device__ __forceinline__ void load_vel(const void *base, float scale, int64_t n, typename VelT<MODE>::T out[3]) {
    if constexpr (MODE == P_F64) {
        double4 v = reinterpret_cast<const double4 *>(base)[n];
        out[0] = v.x;
        out[1] = v.y;
        out[2] = v.z;
    } else if constexpr (MODE == P_F32) {
        float4 v = reinterpret_cast<const float4 *>(base)[n];
        out[0] = v.x;
        out[1] = v.y;
        out[2] = v.z;
    } else {
        uint2 w = reinterpret_cast<const uint2 *>(base)[n];
        unsigned short h0 = (unsigned short)(w.x & 0xffffu), h1 = (unsigned short)(w.x >> 16);
        unsigned short h2 = (unsigned short)(w.y & 0xffffu);
        if constexpr (MODE == P_BF16) {
            out[0] = __uint_as_float((unsigned)h0 << 16) * scale;
            out[1] = __uint_as_float((unsigned)h1 << 16) * scale;
            out[2] = __uint_as_float((unsigned)h2 << 16) * scale;
        } else {
            out[0] = __half2float(__ushort_as_half(h0)) * scale;
            out[1] = __half2float(__ushort_as_half(h1)) * scale;
            out[2] = __half2float(__ushort_as_half(h2)) * scale;
        }
    }
}

/* ------------------------------------------------------------------------ */
/* unstructured interpolation (ompVC/velocity.c:459-621)                     */
/* ------------------------------------------------------------------------ */
/* Probe state: element (walk start, updated in place) and a left flag. */
struct Probe {
    int elem;
    int left;
};

template <int MODE, int DIM>
__device__ __forceinline__ void interp_unstruct(const DevMesh &m, const DevField &f, double tloc, int e, double r,
                                                double s, double t, double out[3]);

/* reduced-precision modes: velocities of an element's nodes in the two
 * bound slices as loaded (FP32 values, or 16-bit words before scaling), so
 * the gather can be issued before the containment test that decides whether
 * it is used */
struct F3 {
    float x, y, z;
};

/* What a lane has stored in its LDS rows is read from there below this point
 * also by the lanes that stored it: taken from their registers instead, the
 * whole element would have to stay live beside the rows' copy. */
__device__ __forceinline__ void reload_rows() { asm volatile("" ::: "memory"); }

template <int MODE, int DIM>
struct NodeVel {
    static constexpr int NN = DIM == 3 ? 4 : 3;
    typename std::conditional<MODE == P_F32, F3, uint2>::type lo[NN], hi[NN];
};

template <int MODE>
__device__ __forceinline__ void ld_vel_word(const void *base, uint32_t n, F3 &w) {
    const float4 v = ld32(reinterpret_cast<const float4 *>(base), n);
    w.x = v.x;
    w.y = v.y;
    w.z = v.z;
}

template <int MODE>
__device__ __forceinline__ void ld_vel_word(const void *base, uint32_t n, uint2 &w) {
    w = ld32(reinterpret_cast<const uint2 *>(base), n);
}

template <int MODE, int DIM>
__device__ __forceinline__ void gather_vel(const DevField &f, int4 nd, NodeVel<MODE, DIM> &g) {
    const uint32_t ids[4] = {(uint32_t)nd.x, (uint32_t)nd.y, (uint32_t)nd.z, (uint32_t)nd.w};
    for (int q = 0; q < NodeVel<MODE, DIM>::NN; q++) {
        ld_vel_word<MODE>(f.lo, ids[q], g.lo[q]);
        ld_vel_word<MODE>(f.hi, ids[q], g.hi[q]);
    }
}

template <int MODE>
__device__ __forceinline__ void node_comp(const F3 &w, float v[3]) {
    v[0] = w.x;
    v[1] = w.y;
    v[2] = w.z;
}

template <int MODE>
__device__ __forceinline__ void node_comp(const uint2 &w, float v[3]) {
    const unsigned short h0 = (unsigned short)(w.x & 0xffffu), h1 = (unsigned short)(w.x >> 16);
    const unsigned short h2 = (unsigned short)(w.y & 0xffffu);
    if constexpr (MODE == P_BF16) {
        v[0] = __uint_as_float((unsigned)h0 << 16);
        v[1] = __uint_as_float((unsigned)h1 << 16);
        v[2] = __uint_as_float((unsigned)h2 << 16);
    } else {
        v[0] = __half2float(__ushort_as_half(h0));
        v[1] = __half2float(__ushort_as_half(h1));
        v[2] = __half2float(__ushort_as_half(h2));
    }
}

/* the reference's weights fabs(r), fabs(s), fabs(t) and 1 minus their sum
 * (velocity.c:574-581, n0 + (n1-n0)|r| + (n2-n0)|s| + (n3-n0)|t|) applied to
 * each slice, then the time weights (1 - tl) and tl, which carry the 16-bit
 * slices' scales; FP32 throughout */
template <int MODE, int DIM>
__device__ __forceinline__ void interp_gathered(const DevField &f, const NodeVel<MODE, DIM> &g, float tl, float r,
                                                float s, float t, float out[3]) {
#pragma clang fp contract(off)
    constexpr int NN = NodeVel<MODE, DIM>::NN;
    float w[4];
    w[1] = fabsf(r);
    w[2] = fabsf(s);
    w[3] = DIM == 3 ? fabsf(t) : 0.0f;
    w[0] = DIM == 3 ? ((1.0f - w[1]) - w[2]) - w[3] : (1.0f - w[1]) - w[2];
    float lo[3], hi[3];
    for (int q = 0; q < NN; q++) {
        float a[3], b[3];
        node_comp<MODE>(g.lo[q], a);
        node_comp<MODE>(g.hi[q], b);
        for (int c = 0; c < 3; c++) {
            lo[c] = q == 0 ? w[0] * a[c] : __builtin_fmaf(w[q], a[c], lo[c]);
            hi[c] = q == 0 ? w[0] * b[c] : __builtin_fmaf(w[q], b[c], hi[c]);
        }
    }
    const float tlo = MODE == P_F32 ? 1.0f - tl : (1.0f - tl) * f.scale_lo;
    const float thi = MODE == P_F32 ? tl : tl * f.scale_hi;
    for (int c = 0; c < 3; c++) out[c] = (DIM == 2 && c == 2) ? 0.0f : __builtin_fmaf(thi, hi[c], tlo * lo[c]);
}

template <int MODE, int DIM>
__device__ __forceinline__ void interp_nodes_f(const DevField &f, float tl, int4 nd, float r, float s, float t,
                                               float out[3]) {
    NodeVel<MODE, DIM> g;
    gather_vel<MODE, DIM>(f, nd, g);
    interp_gathered<MODE, DIM>(f, g, tl, r, s, t, out);
}

template <int MODE, int DIM>
__device__ __forceinline__ void interp_unstruct_f(const DevMesh &m, const DevField &f, float tl, int e, float r,
                                                  float s, float t, float out[3]) {
    interp_nodes_f<MODE, DIM>(f, tl, ld32(m.conn, e), r, s, t, out);
}

template <int MODE, int DIM>
__device__ __forceinline__ void vel_unstruct(const DevMesh &m, const DevField &f, double tloc, double x, double y,
                                             double z, Probe &p, double out[3], int &err) {
    if (p.elem < 0 || p.elem >= m.ne) {
        err = E_ELEM;
        out[0] = out[1] = out[2] = 0.0;
        return;
    }
    double r, s, t;
    int e = walk<MODE, DIM>(m, x, y, z, p.elem, ACC_INTERP, r, s, t, err);
    if (e == -2) {
        out[0] = out[1] = out[2] = 0.0;
        return;
    }
    if (e == -1) {
        p.elem = -1;
        p.left = 1;
        out[0] = out[1] = out[2] = 0.0;
        return;
    }
    p.elem = e;
    interp_unstruct<MODE, DIM>(m, f, tloc, e, r, s, t, out);
}

/* velocity at natural coordinates (r,s,t) of element e (velocity.c:603-619) */
template <int MODE, int DIM>
__device__ __forceinline__ void interp_unstruct(const DevMesh &m, const DevField &f, double tloc, int e, double r,
                                                double s, double t, double out[3]) {
    int4 nd = ld32(m.conn, e);
    using VT = typename VelT<MODE>::T;
    if constexpr (MODE == P_F64) {
#pragma clang fp contract(off)
        double a[4][3], b[4][3], n[4][3];
        const int nn = DIM == 3 ? 4 : 3;
        int ids[4] = {nd.x, nd.y, nd.z, nd.w};
        for (int q = 0; q < nn; q++) {
            load_vel_node<MODE>(f.lo, 1.0f, ids[q], a[q]);
            load_vel_node<MODE>(f.hi, 1.0f, ids[q], b[q]);
            for (int c = 0; c < 3; c++) n[q][c] = (1 - tloc) * a[q][c] + tloc * b[q][c];
        }
        double ar = fabs(r), as = fabs(s), at = fabs(t);
        if (DIM == 3) {
            for (int c = 0; c < 3; c++)
                out[c] = n[0][c] + (n[1][c] - n[0][c]) * ar + (n[2][c] - n[0][c]) * as + (n[3][c] - n[0][c]) * at;
        } else {
            for (int c = 0; c < 2; c++) out[c] = n[0][c] + (n[1][c] - n[0][c]) * ar + (n[2][c] - n[0][c]) * as;
            out[2] = 0.0;
        }
    } else {
        float v[3];
        interp_unstruct_f<MODE, DIM>(m, f, (float)tloc, e, (float)r, (float)s, (float)t, v);
        for (int c = 0; c < 3; c++) out[c] = v[c];
    }
}

/* ------------------------------------------------------------------------ */
/* Cartesian domain tests and interpolation (ompVC/velocity.c:257-457,624-669) */
/* ------------------------------------------------------------------------ */
__device__ __forceinline__ int outside_domain(const DevMesh &m, double x, double y, double z) {
#pragma clang fp contract(off)
    if (x < (m.bounds[0] - TINY) || x > (m.bounds[1] + TINY)) return 1;
    if (y < (m.bounds[2] - TINY) || y > (m.bounds[3] + TINY)) return 1;
    if (z < (m.bounds[4] - TINY) || z > (m.bounds[5] + TINY)) return 1;
    return 0;
}

/* (t - tmin) / (tmax - tmin), tinv = fvc_near_inverse(tmax - tmin) */
__device__ __forceinline__ double time_loc(const DevField &f, double t, double tinv) {
#pragma clang fp contract(off)
    const double d = t - f.tmin, span = f.tmax - f.tmin;
    return tinv != 0.0 ? fvc_div_near(d, span, tinv) : d / span;
}

/* x / 6 of the RK4 increment; infinities take the division.  The three
 * quotients side by side: each is a chain of five dependent instructions. */
__device__ __forceinline__ void sixths(double x[3]) {
    if (fmax(fabs(x[0]), fmax(fabs(x[1]), fabs(x[2]))) < 1e300) {
        for (int c = 0; c < 3; c++) x[c] = fvc_div_near(x[c], 6.0, 1.0 / 6.0);
    } else {
        for (int c = 0; c < 3; c++) x[c] = x[c] / 6;
    }
}

/* Cell and local coordinates of X in the velocity grid, false outside it
 * (velocity.c:257-457): q = (X - min) / del, outside where floor(q) < 0 or
 * ceil(q) > res - 1, which for an integer bound is q < 0 or q > res - 1.
 * The axes are computed side by side, without a branch between them. */
template <int DIM>
__device__ __forceinline__ bool cart_cell(const DevMesh &m, const double X[3], int cell[3], double loc[3]) {
#pragma clang fp contract(off)
    bool in = true, near = true;
    double d[DIM], q[DIM], r[DIM];
    for (int a = 0; a < DIM; a++) {
        d[a] = X[a] - m.cmin[a];
        near = near && m.cinv[a] != 0.0;
    }
    if (near)
        for (int a = 0; a < DIM; a++) q[a] = fvc_div_near(d[a], m.cdel[a], m.cinv[a]);
    else
        for (int a = 0; a < DIM; a++) q[a] = d[a] / m.cdel[a];
    for (int a = 0; a < DIM; a++) {
        const double top = (double)(m.cres[a] - 1);
        in = in && !(q[a] < 0.0) && !(q[a] > top) && !(fabs(d[a]) >= m.cfar[a]);
        const double fl = floor(q[a]);
        r[a] = d[a] - fl * m.cdel[a];
        cell[a] = (int)fl;
    }
    if (near)
        for (int a = 0; a < DIM; a++) r[a] = fvc_div_near(r[a], m.cdel[a], m.cinv[a]);
    else
        for (int a = 0; a < DIM; a++) r[a] = r[a] / m.cdel[a];
    for (int a = 0; a < DIM; a++) { /* the last node belongs to the last cell */
        const bool end = cell[a] == m.cres[a] - 1;
        loc[a] = end ? 1.0 : r[a];
        cell[a] = end ? cell[a] - 1 : cell[a];
    }
    return in;
}

/* The corners of a cell, (x, y, z) offsets in the bits (4, 2, 1) of the
 * corner number; a 2-D cell's are 0, 2, 4 and 6. */
template <int MODE, int DIM>
struct CartCorners {
    static constexpr int NQ = 1 << DIM, STEP = DIM == 3 ? 1 : 2;
    static constexpr int STRIDE = MODE == P_F64 ? 32 : MODE == P_F32 ? 16 : 8;
    const char *row[4]; /* corners (0, y, z), index 2 y + z; corner x + 1 follows at STRIDE */
    __device__ __forceinline__ void at(const DevMesh &m, const void *base, int64_t c0) {
        const int64_t nx = m.cres[0] * (int64_t)STRIDE;
        row[0] = (const char *)base + c0 * STRIDE;
        row[2] = row[0] + nx;
        if (DIM == 3) {
            row[1] = row[0] + nx * m.cres[1];
            row[3] = row[1] + nx;
        }
    }
    __device__ __forceinline__ const char *corner(int q) const { return row[q & 3] + (q >> 2) * STRIDE; }
};

template <int DIM>
__device__ __forceinline__ int64_t cart_index(const DevMesh &m, const int cell[3]) {
    const int64_t row = DIM == 3 ? (int64_t)cell[2] * m.cres[1] + cell[1] : (int64_t)cell[1];
    return row * m.cres[0] + cell[0];
}

/* LDS rows of the Cartesian RK4 kernels: the corner velocities of the cell a
 * lane interpolated in last (both slices), as SmRows holds an element's.  A
 * stage moves a fraction of a cell, so gathering only after a change of cell
 * cuts the gathers several times over.  In FP64 only in 2-D, for slices whose
 * third component is zero: a 3-D cell is 384 bytes, which would leave 6 waves
 * on a CU.  300,007 points in random order on an 80x64x48 grid, FP32, 20
 * steps: 2,244 us, bound by the lines those gathers pull through the L2, to
 * 265 us. */
template <int MODE, int DIM>
struct CartRows {
    static constexpr int NQ = 1 << DIM, W = MODE == P_F64 ? 4 : MODE == P_F32 ? DIM : 2;
    static constexpr int N = MODE == P_F64 && DIM == 3 ? 0 : (2 * NQ * W + 3) / 4;
};

/* this lane's last cell and its rows (rows null: gather every time) */
struct CartLast {
    float4 *rows = nullptr;
    int64_t cell = -1;
};

template <int DIM>
__device__ __forceinline__ void cart_velocity_f64(const DevMesh &m, const DevField &f, double tl, const int cell[3],
                                                  const double loc[3], CartLast &last, double out[3]) {
#pragma clang fp contract(off)
    using C = CartCorners<P_F64, DIM>;
    const int64_t c0 = cart_index<DIM>(m, cell);
    const double tw[2] = {1 - tl, tl};
    /* a corner's weight: products left to right, time, x, y, z */
    auto weight = [&](int s, int q) {
        double w = tw[s] * ((q & 4) ? loc[0] : (1 - loc[0])) * ((q & 2) ? loc[1] : (1 - loc[1]));
        if (DIM == 3) w = w * ((q & 1) ? loc[2] : (1 - loc[2]));
        return w;
    };
    double acc[3] = {0.0, 0.0, 0.0};
    if (DIM == 2 && !f.vals && last.rows) { /* finite, third component zero */
        if (c0 != last.cell) {
            C cc[2];
            cc[0].at(m, f.lo, c0);
            cc[1].at(m, f.hi, c0);
            for (int k = 0; k < 8; k++)
                last.rows[64 * k] = *reinterpret_cast<const float4 *>(cc[k >> 2].corner((k & 3) * 2));
            last.cell = c0;
        }
        reload_rows();
        for (int s = 0; s < 2; s++)
            for (int k = 0; k < 4; k++) {
                const double2 v = *reinterpret_cast<const double2 *>(last.rows + 64 * (4 * s + k));
                const double w = weight(s, 2 * k);
                acc[0] = s == 0 && k == 0 ? v.x * w : acc[0] + v.x * w;
                acc[1] = s == 0 && k == 0 ? v.y * w : acc[1] + v.y * w;
            }
        for (int c = 0; c < 3; c++) out[c] = acc[c];
        return;
    }
    double big[3] = {0.0, 0.0, 0.0};
#pragma unroll 1 /* both slices' corners at once spill */
    for (int s = 0; s < 2; s++) {
        C cc;
        cc.at(m, s ? f.hi : f.lo, c0);
        double v[8][3];
        for (int q = 0; q < 8; q += C::STEP) {
            const double *p = reinterpret_cast<const double *>(cc.corner(q));
            for (int c = 0; c < 3; c++) v[q][c] = p[c];
        }
        for (int q = 0; q < 8; q += C::STEP) {
            const double w = weight(s, q);
            for (int c = 0; c < 3; c++) acc[c] = s == 0 && q == 0 ? v[q][c] * w : acc[c] + v[q][c] * w;
        }
        /* In 2-D the reference's formula also adds every corner of the plane
         * k + 1, the same node, with weight zero: nothing, unless the node
         * holds an infinity. */
        if (DIM == 2 && (f.vals & VALS_INF))
            for (int q = 0; q < 8; q += C::STEP)
                for (int c = 0; c < 3; c++) big[c] = fmax(big[c], fabs(v[q][c]));
    }
    if (DIM == 2 && (f.vals & VALS_INF))
        for (int c = 0; c < 3; c++) acc[c] = acc[c] + big[c] * 0.0;
    for (int c = 0; c < 3; c++) out[c] = acc[c];
}

/* one corner's words as loaded: FP32 components, or four 16-bit values */
template <int MODE, int DIM>
__device__ __forceinline__ void cart_words(const char *p, float *w) {
    if constexpr (MODE == P_F32) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        w[0] = v.x;
        w[1] = v.y;
        if (DIM == 3) w[2] = v.z;
    } else {
        const uint2 v = *reinterpret_cast<const uint2 *>(p);
        w[0] = __uint_as_float(v.x);
        w[1] = __uint_as_float(v.y);
    }
}

template <int MODE, int DIM>
__device__ __forceinline__ void cart_value(const float *w, float scale, float v[3]) {
    if constexpr (MODE == P_F32) {
        v[0] = w[0];
        v[1] = w[1];
        v[2] = DIM == 3 ? w[2] : 0.0f;
    } else {
        node_comp<MODE>(make_uint2(__float_as_uint(w[0]), __float_as_uint(w[1])), v);
        for (int c = 0; c < 3; c++) v[c] = v[c] * scale;
    }
}

template <int MODE, int DIM>
__device__ __forceinline__ void cart_interp_f32(const DevField &f, const float *w, double tloc, const double loc[3],
                                                double out[3]) {
#pragma clang fp contract(off)
    using C = CartCorners<MODE, DIM>;
    using R = CartRows<MODE, DIM>;
    const float tl = (float)tloc, xl = (float)loc[0], yl = (float)loc[1], zl = (float)loc[2];
    float acc[3] = {0.f, 0.f, 0.f};
    for (int k = 0; k < R::NQ; k++) {
        const int q = k * C::STEP;
        const float wx = (q & 4) ? xl : (1.f - xl), wy = (q & 2) ? yl : (1.f - yl);
        float g = wx * wy;
        if (DIM == 3) g = g * ((q & 1) ? zl : (1.f - zl));
        float a[3], b[3];
        cart_value<MODE, DIM>(w + 2 * R::W * k, f.scale_lo, a);
        cart_value<MODE, DIM>(w + 2 * R::W * k + R::W, f.scale_hi, b);
        for (int c = 0; c < 3; c++) acc[c] += g * (a[c] + tl * (b[c] - a[c]));
    }
    out[0] = acc[0];
    out[1] = acc[1];
    out[2] = DIM == 3 ? (double)acc[2] : 0.0;
}

template <int MODE, int DIM>
__device__ __forceinline__ void cart_velocity_f32(const DevMesh &m, const DevField &f, double tloc, const int cell[3],
                                                  const double loc[3], CartLast &last, double out[3]) {
#pragma clang fp contract(off)
    using C = CartCorners<MODE, DIM>;
    using R = CartRows<MODE, DIM>;
    const int64_t c0 = cart_index<DIM>(m, cell);
    /* corner by corner: the lo slice's words, then the hi slice's */
    if (!last.rows || c0 != last.cell) {
        float w[4 * R::N];
        C lo, hi;
        lo.at(m, f.lo, c0);
        hi.at(m, f.hi, c0);
        /* Corner x + 1 right after corner x, one line apart at most: between
         * them the other rows' lines, 64 each, would push theirs out of the
         * L1 (2-D, 150,000 random points: L1 misses 5.3e7 against 3.1e7 a
         * launch). */
        for (int q = 0; q < R::NQ / 2; q++)
            for (int x = 0; x < 2; x++) {
                const int k = q + x * R::NQ / 2;
                cart_words<MODE, DIM>(lo.corner(k * C::STEP), w + 2 * R::W * k);
            }
        for (int q = 0; q < R::NQ / 2; q++)
            for (int x = 0; x < 2; x++) {
                const int k = q + x * R::NQ / 2;
                cart_words<MODE, DIM>(hi.corner(k * C::STEP), w + 2 * R::W * k + R::W);
            }
        if (!last.rows) {
            cart_interp_f32<MODE, DIM>(f, w, tloc, loc, out);
            return;
        }
        for (int k = 0; k < R::N; k++)
            last.rows[64 * k] = make_float4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
        last.cell = c0;
    }
    reload_rows();
    float w[4 * R::N];
    for (int k = 0; k < R::N; k++) {
        const float4 v = last.rows[64 * k];
        w[4 * k] = v.x;
        w[4 * k + 1] = v.y;
        w[4 * k + 2] = v.z;
        w[4 * k + 3] = v.w;
    }
    cart_interp_f32<MODE, DIM>(f, w, tloc, loc, out);
}

/* velocity at a position inside the velocity grid */
template <int MODE, int DIM>
__device__ __forceinline__ void cart_velocity(const DevMesh &m, const DevField &f, double tloc, const int cell[3],
                                              const double loc[3], CartLast &last, double out[3]) {
    if constexpr (MODE == P_F64) cart_velocity_f64<DIM>(m, f, tloc, cell, loc, last, out);
    else cart_velocity_f32<MODE, DIM>(m, f, tloc, cell, loc, last, out);
}

/* ------------------------------------------------------------------------ */
/* particle state and integrators (ompVC/integration.c)                     */
/* ------------------------------------------------------------------------ */
struct PState {
    double X[3];
    double V[3];
    int elem;
    int left;
    double left_time;
    /* multistep history: velocities at the two previous nodes, count held */
    double F1[3], F2[3];
    int nhist;
    double scalar; /* activation potential */
};

__device__ __forceinline__ double sign_of(double a, double b) { return b >= 0.0 ? fabs(a) : -fabs(a); }

/* GetVelocity on the particle itself (side effects on elem / left). */
template <int MODE, int DIM>
__device__ __forceinline__ void get_velocity(const DevMesh &m, const DevField &f, double tq, PState &p, double out[3],
                                             int &err) {
#pragma clang fp contract(off)
    double tloc = (tq - f.tmin) / (f.tmax - f.tmin);
    if (m.mesh_type == 1) {
        if (p.elem < 0 || p.elem >= m.ne) {
            err = E_ELEM;
            return;
        }
        if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
            err = E_TLOC;
            return;
        }
        Probe pr{p.elem, p.left};
        vel_unstruct<MODE, DIM>(m, f, tloc, p.X[0], p.X[1], p.X[2], pr, out, err);
        p.elem = pr.elem;
        p.left = pr.left;
    } else {
        int cell[3];
        double loc[3];
        if (!cart_cell<DIM>(m, p.X, cell, loc)) {
            out[0] = out[1] = out[2] = 0.0;
            p.left = 1;
            return;
        }
        if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
            err = E_TLOC;
            return;
        }
        CartLast none;
        cart_velocity<MODE, DIM>(m, f, tloc, cell, loc, none, out);
    }
}

/* velocity at a probe position for a stage (probe owns its element / flag) */
template <int MODE, int DIM, int UNSTRUCT>
__device__ __forceinline__ void stage_velocity(const DevMesh &m, const DevField &f, double tq, const double X[3],
                                               Probe &pr, double out[3], int &err, double tinv, CartLast &last) {
#pragma clang fp contract(off)
    const double tloc = time_loc(f, tq, tinv);
    if (UNSTRUCT) {
        if (pr.elem == -1) {
            err = E_ELEM;
            return;
        }
        if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
            err = E_TLOC;
            return;
        }
        vel_unstruct<MODE, DIM>(m, f, tloc, X[0], X[1], X[2], pr, out, err);
    } else {
        int cell[3];
        double loc[3];
        if (!cart_cell<DIM>(m, X, cell, loc)) {
            out[0] = out[1] = out[2] = 0.0;
            pr.left = 1;
            return;
        }
        if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
            err = E_TLOC;
            return;
        }
        cart_velocity<MODE, DIM>(m, f, tloc, cell, loc, last, out);
    }
}

/* Reduced-precision modes on unstructured meshes: the stage velocity at an
 * FP32 probe (anchor A, offset d; the point (centre + A) + d) and at the
 * FP64 position X, with FP32 results. */
template <int MODE, int DIM>
__device__ __forceinline__ void stage_velocity_c(const DevMesh &m, const DevField &f, double tloc, const float A[3],
                                                 const float d[3], Probe &pr, float out[3], int &err) {
#pragma clang fp contract(off)
    out[0] = out[1] = out[2] = 0.0f;
    if (pr.elem == -1) {
        err = E_ELEM;
        return;
    }
    if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
        err = E_TLOC;
        return;
    }
    if (pr.elem < 0 || pr.elem >= m.ne) {
        err = E_ELEM;
        return;
    }
    float r, s, t;
    int4 nd;
    const int e = walk_c<DIM>(m, A, d, pr.elem, ACC_INTERP, r, s, t, nd, err);
    if (e == -2) return;
    if (e == -1) {
        pr.elem = -1;
        pr.left = 1;
        return;
    }
    pr.elem = e;
    interp_nodes_f<MODE, DIM>(f, (float)tloc, nd, r, s, t, out);
}

template <int MODE, int DIM>
__device__ __forceinline__ void stage_velocity_x(const DevMesh &m, const DevField &f, double tloc, const double X[3],
                                                 Probe &pr, float out[3], int &err) {
#pragma clang fp contract(off)
    out[0] = out[1] = out[2] = 0.0f;
    if (pr.elem == -1) {
        err = E_ELEM;
        return;
    }
    if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
        err = E_TLOC;
        return;
    }
    if (pr.elem < 0 || pr.elem >= m.ne) {
        err = E_ELEM;
        return;
    }
    double r, s, t;
    const int e = walk<MODE, DIM>(m, X[0], X[1], X[2], pr.elem, ACC_INTERP, r, s, t, err);
    if (e == -2) return;
    if (e == -1) {
        pr.elem = -1;
        pr.left = 1;
        return;
    }
    pr.elem = e;
    interp_unstruct_f<MODE, DIM>(m, f, (float)tloc, e, (float)r, (float)s, (float)t, out);
}

/* ------------------------------------------------------------------------ */
/* Resumable integration of one interval [a, b]: one Advect call of the      */
/* reference.  IState keeps what the reference keeps in locals across its    */
/* step loop: the current time, the step size (which stays clipped once      */
/* clipped, integration.c:346-352), and the four RK4 stage probes, each with */
/* its own walk element and left flag (integration.c:337-341).  With         */
/* max_steps unlimited this is the reference's loop; with a budget, a        */
/* persistent kernel can stop and resume it with identical arithmetic.       */
/* ------------------------------------------------------------------------ */
struct IState {
    double tc, h;
    Probe mp[4];
    int started;
};

enum { INT_EULER = 0, INT_RK4 = 1, INT_RKF = 2, INT_AB2 = 3, INT_AB3 = 4 };

/* Strain rate at the point (GetStrainRate_Unstructured, ompVC/strainrate.c:
 * 232-246; GetStrainRate_Cartesian, :196-230), linear in time between the two
 * loaded strain-rate slices.  Unstructured: the reference first walks from
 * the point's element (search acceptance, d > -TINY); the element held here
 * was located by that same acceptance at this same position (the step's
 * final locate, the seed chain or a launch walk that keeps it), so that walk
 * returns it unchanged and is not repeated. */
/* Exposure-time sums are kept exactly: a time t >= 0 adds floor(t 2^CET_FRAC)
 * to a 128-bit fixed-point accumulator (two 64-bit words, the carry of the low
 * word added to the high one), so the per-element totals do not depend on the
 * order in which the parallel steps arrive; the reference adds in its
 * threads' arrival order (exposuretime.c:135-164). */
constexpr int CET_FRAC = 100;

__device__ inline void cet_add(unsigned long long *lo, unsigned long long *hi, double v) {
    if (!(v > 0.0)) return;
    int e;
    const double fr = frexp(v, &e);                            /* v = fr 2^e, fr in [0.5, 1) */
    const unsigned long long mnt = (unsigned long long)ldexp(fr, 53); /* v = mnt 2^(e-53) */
    const int sh = e - 53 + CET_FRAC;
    unsigned long long l = 0, h = 0;
    if (sh <= -64) return;
    if (sh < 0) l = mnt >> (-sh);
    else if (sh < 64) {
        l = mnt << sh;
        h = sh ? (mnt >> (64 - sh)) : 0ull;
    } else if (sh < 128) {
        h = mnt << (sh - 64);
    }
    const unsigned long long old = atomicAdd(lo, l);
    const unsigned long long carry = (old + l < old) ? 1ull : 0ull;
    if (h + carry) atomicAdd(hi, h + carry);
}

/* ComputeExposureTime (exposuretime.c:120-178) for a step from X0 to X1 of
 * length h, X1 in element e1: the whole step to the element of X0 if that is
 * e1, else h/(S-1) to the element of each of the S-1 points X0 + a (X1 - X0),
 * a = s/(S-1), s = 1..S-1, walking from point to point, with an encounter
 * where the element changes; points in no element are skipped. */
template <int DIM>
__device__ inline void cet_step(const DevMesh &m, const DevField &f, const double X0[3], const double X1[3], int e1,
                                double h, int &err) {
#pragma clang fp contract(off)
    int e0 = local_search<DIM>(m, X0[0], X0[1], X0[2], e1, err);
    if (err) return;
    if (e0 < 0) {
        e0 = hash_global<DIM>(m, X0[0], X0[1], X0[2]);
        if (e0 < 0) {
            err = E_CET;
            return;
        }
    }
    if (e0 == e1) {
        cet_add(f.cet_lo + e0, f.cet_hi + e0, h);
        return;
    }
    const int S = f.cet_sub;
    int last = e0;
    for (int s = 1; s < S; s++) {
        const double a = ((double)s) / ((double)(S - 1));
        double Xt[3];
        for (int i = 0; i < 3; i++) Xt[i] = (1 - a) * X0[i] + a * X1[i];
        int et = local_search<DIM>(m, Xt[0], Xt[1], Xt[2], last, err);
        if (err) return;
        if (et < 0) {
            et = hash_global<DIM>(m, Xt[0], Xt[1], Xt[2]);
            if (et < 0) continue; /* path crosses the outside: no contribution (exposuretime.c:160-165) */
        }
        cet_add(f.cet_lo + et, f.cet_hi + et, h / (S - 1));
        if (et != last) {
            atomicAdd(f.cet_enc + et, 1);
            last = et;
        }
    }
}

template <int DIM, int UNSTRUCT>
__device__ inline double strain_rate(const DevMesh &m, const DevField &f, double t, const PState &p, int &err) {
#pragma clang fp contract(off)
    const double tloc = (t - f.tmin) / (f.tmax - f.tmin);
    if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
        err = E_TLOC;
        return 0.0;
    }
    int64_t idx;
    if (UNSTRUCT) {
        if (p.elem < 0 || p.elem >= m.ne) {
            err = E_ELEM;
            return 0.0;
        }
        idx = p.elem;
    } else {
        if (outside_domain(m, p.X[0], p.X[1], p.X[2])) {
            err = E_LEFT;
            return 0.0;
        }
        int cell[3] = {0, 0, 0};
        for (int a = 0; a < DIM; a++) {
            cell[a] = (int)floor((p.X[a] - m.cmin[a]) / m.cdel[a]);
            if (cell[a] == m.cres[a] - 1) cell[a] = m.cres[a] - 2;
            if (cell[a] < 0 || cell[a] > m.cres[a] - 2) { /* the reference asserts here */
                err = E_ELEM;
                return 0.0;
            }
        }
        const int64_t imax = m.cres[0] - 1, jmax = m.cres[1] - 1;
        idx = ((int64_t)cell[2] * jmax + cell[1]) * imax + cell[0];
    }
    return (1 - tloc) * f.sr_lo[idx] + tloc * f.sr_hi[idx];
}


/* ------------------------------------------------------------------------ */
/* RK4 of the reduced-precision modes on unstructured meshes, one           */
/* containment test per lane per loop iteration                              */
/* ------------------------------------------------------------------------ */
/* The same integrator as interval_run's RK4 (integration.c:317-462): four
 * stage probes that keep their own walk elements, the increment
 * h (f0 + 2 k2 + 2 k3 + k4) / 6, a locate walk at the new position, the exit
 * revert, the first stage taking the locate's element and coordinates.  It is
 * written as a state machine: a lane is in one of five phases (first-stage
 * walk at X, the k2, k3, k4 probe walks, the locate walk), and each pass of
 * the loop makes one containment test for every lane, followed by the
 * interpolation of the lanes whose test accepted and the bookkeeping of their
 * next phase.  Walks of different lengths then overlap instead of making the
 * whole wavefront repeat the longest one.  Every lane performs the same
 * floating-point operations, in the same order, as a straight-line walk would.
 * Query points are anchored FP32 offsets (A, d), see nat_fast_c; an
 * undecided test of the first-stage or locate walk is decided in FP64 at the
 * double position X, a probe's at (centre + A) + d. */
enum { PH_F0 = 0, PH_K2 = 1, PH_K3 = 2, PH_K4 = 3, PH_LOC = 4, PH_DONE = 5 };

/* Per-lane rows of LDS holding the frame of the element a lane tested last
 * and the node velocities (both slices) of the element it interpolated in
 * last; row k of lane l is at [64 k + l], so a wave's 16-byte accesses are
 * contiguous.
 * Why: gathered anew, a pass costs 13 per-lane gathers (frame, connectivity,
 * eight node velocities), and their tag look-ups kept the L1 busy 94% of the
 * cycles (1.1-1.2 look-ups per CU and cycle, 32 per particle-step) with the
 * vector ALUs at 64-68%; but a probe moves a tenth of an element per step, so
 * nearly every pass asks for what the lane had in the pass before.  With the
 * rows only lanes whose element changed gather: 5.1-5.5 look-ups per step,
 * vector ALUs 77-80% busy.  k_advect (4M tracers, 20 steps, 5.6M tets) 3.44 -> 2.76
 * ms a launch, k_ftle_advect (96x96x480 points) 4.49 -> 2.66 ms, the RK4
 * class of a batch 2.1 -> 1.2 ms.  LDS and not registers: held in registers
 * (40 more) the kernels spill 56-64 at 4 waves per SIMD.  160 bytes a lane
 * in FP32 is the whole LDS at 4 waves per SIMD (16 waves of 10 KB), which is
 * why nothing else of these kernels lies there. */
template <int MODE, int DIM>
struct SmRows {
    static constexpr int NN = DIM == 3 ? 4 : 3;
    static constexpr int FRAME = DIM == 3 ? 4 : 3;
    static constexpr int VEL = (NN * (MODE == P_F32 ? 6 : 4) + 3) / 4;
    static constexpr int N = MODE == P_F64 ? NN * DIM : FRAME + VEL; /* FP64: velocities only (rk4_sm64) */
};

/* GEN, the build of interval_run that a kernel compiles:
 *   0  RK4 without extrapolation, strain rate or exposure time, with LDS rows:
 *      rk4_sm, rk4_sm64, rk4_cart
 *   1  every integrator and option, straight-line walks
 *   2  AB2 and AB3 without those options on rk4_sm (reduced precision,
 *      unstructured)
 *   3  RK4 with straight-line walks (FP64, unstructured)
 * Where two of them can run, they give the same bits. */
/* rows per lane of the kernels that have them, and this lane's in a block of
 * BS lanes (null where there are none) */
template <int MODE, int DIM, int UNS, int GEN>
constexpr int lane_rows() {
    return GEN == 1 || GEN == 3 ? 0 : UNS ? SmRows<MODE, DIM>::N : CartRows<MODE, DIM>::N;
}

template <int MODE, int DIM, int UNS, int GEN, int BS>
__device__ __forceinline__ float4 *sm_rows() {
    constexpr int N = lane_rows<MODE, DIM, UNS, GEN>();
    if constexpr (N > 0) {
        __shared__ float4 s_rows[N * BS];
        return s_rows + (threadIdx.x >> 6) * (64 * N) + (threadIdx.x & 63);
    } else {
        return nullptr;
    }
}

template <int MODE, int DIM>
__device__ __forceinline__ void vel_to_rows(const NodeVel<MODE, DIM> &g, float4 *rows) {
    constexpr int NN = NodeVel<MODE, DIM>::NN, W = MODE == P_F32 ? 6 : 4;
    float w[4 * SmRows<MODE, DIM>::VEL] = {};
    for (int q = 0; q < NN; q++) {
        if constexpr (MODE == P_F32) {
            w[W * q] = g.lo[q].x;
            w[W * q + 1] = g.lo[q].y;
            w[W * q + 2] = g.lo[q].z;
            w[W * q + 3] = g.hi[q].x;
            w[W * q + 4] = g.hi[q].y;
            w[W * q + 5] = g.hi[q].z;
        } else {
            w[W * q] = __uint_as_float(g.lo[q].x);
            w[W * q + 1] = __uint_as_float(g.lo[q].y);
            w[W * q + 2] = __uint_as_float(g.hi[q].x);
            w[W * q + 3] = __uint_as_float(g.hi[q].y);
        }
    }
    for (int k = 0; k < SmRows<MODE, DIM>::VEL; k++)
        rows[64 * k] = make_float4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
}

template <int MODE, int DIM>
__device__ __forceinline__ void vel_from_rows(const float4 *rows, NodeVel<MODE, DIM> &g) {
    constexpr int NN = NodeVel<MODE, DIM>::NN, W = MODE == P_F32 ? 6 : 4;
    float w[4 * SmRows<MODE, DIM>::VEL];
    for (int k = 0; k < SmRows<MODE, DIM>::VEL; k++) {
        const float4 v = rows[64 * k];
        w[4 * k] = v.x;
        w[4 * k + 1] = v.y;
        w[4 * k + 2] = v.z;
        w[4 * k + 3] = v.w;
    }
    for (int q = 0; q < NN; q++) {
        if constexpr (MODE == P_F32) {
            g.lo[q] = F3{w[W * q], w[W * q + 1], w[W * q + 2]};
            g.hi[q] = F3{w[W * q + 3], w[W * q + 4], w[W * q + 5]};
        } else {
            g.lo[q] = make_uint2(__float_as_uint(w[W * q]), __float_as_uint(w[W * q + 1]));
            g.hi[q] = make_uint2(__float_as_uint(w[W * q + 2]), __float_as_uint(w[W * q + 3]));
        }
    }
}

/* AB: Adams-Bashforth of the order that itype names, as
 * interval_run defines it, bit for bit: a step is the first stage and the
 * locate walk, whose element and coordinates the next first stage takes, with
 * RK4 steps while the history is short or the step clipped.  Its tests at the
 * position take the FP64 difference to the frame's origin (nat_fast), as the
 * straight-line walks do.  An AB3 class of a batch of 884k particles 1,030 ->
 * 527 us a launch, against the straight-line walks at 2 waves per
 * SIMD (held to 3, the batch kernel spills 45 registers). */
template <int MODE, int DIM, int AB = 0>
__device__ int rk4_sm(const DevMesh &m, const DevField &f, PState &p, IState &is, double a, double b, double dt,
                      int max_steps, int &err, uint32_t &nsteps, double &stop, float4 *rows, int itype = INT_RK4) {
#pragma clang fp contract(off)
    using R = SmRows<MODE, DIM>;
    if (!is.started) {
        if (p.left) {
            err = E_LEFT;
            stop = b;
            return 1;
        }
        if (p.elem < 0 || p.elem >= m.ne) {
            err = E_ELEM;
            stop = b;
            return 1;
        }
        is.tc = a;
        is.h = sign_of(dt, b - a);
        for (int q = 0; q < 4; q++) {
            is.mp[q].elem = p.elem;
            is.mp[q].left = 0;
        }
        is.started = 1;
    }
    const double hmin = 1e-12 * fabs(dt), hfull = sign_of(dt, b - a);
    float f0[3] = {0.f, 0.f, 0.f}; /* AB: the step's first slope */
    bool multi = false;            /* AB: the step is not RK4 */
    const double inv_span = 1.0 / (f.tmax - f.tmin);
    int taken = 0, ret = 1;
    int phase = PH_F0, hops = 0;
    bool tie = false;  /* a test of this locate walk hit d == -TINY */
    bool gone = false; /* a probe of this step left the mesh */
    /* the probes' elements, a ring: q0 is the walk start of the probe whose
     * turn it is (at a step's start and in the locate walk the first stage's) */
    int q0 = is.mp[0].elem, q1 = is.mp[1].elem, q2 = is.mp[2].elem, q3 = is.mp[3].elem;
    /* S: f0, then f0 + 2 k2, f0 + 2 k2 + 2 k3, and from the k4 stage to the
     * locate's end the step's f0 + 2 k2 + 2 k3 + k4 (increment h/6 S) */
    float A[3], D[3], c[3], S[3] = {0.f, 0.f, 0.f}, gc;
    float tl0 = 0.f, tlh = 0.f, tl1 = 0.f; /* time locations of the step's start, middle and end */
    /* anchors of X: A = (float)(X - centre), D its FP32 residual; the walk at
     * X has the offset c = D */
    auto anchor = [&]() {
        for (int k = 0; k < 3; k++) {
            const double xc = p.X[k] - m.centre[k];
            A[k] = (float)xc;
            D[k] = (float)(xc - (double)A[k]);
            c[k] = D[k];
        }
        gc = guard_offset(m, c);
    };
    const int order = itype == INT_AB2 ? 2 : 3;
    /* start of a step (the loop head of integration.c:344); false when the
     * interval is done or the step budget spent */
    auto begin_step = [&]() -> bool {
        if (!((is.tc - b) * (b - a) < 0.0)) {
            stop = b;
            return false;
        }
        if (taken == max_steps) {
            ret = 0;
            return false;
        }
        if ((is.tc + is.h - b) * (is.tc + is.h - a) > 0.0) is.h = sign_of(b - is.tc, b - a);
        const double l0 = (is.tc - f.tmin) * inv_span, l1 = (is.tc + is.h - f.tmin) * inv_span;
        tl0 = (float)l0;
        tlh = (float)((is.tc + is.h / 2 - f.tmin) * inv_span); /* lies between l0 and l1 */
        tl1 = (float)l1;
        if ((l0 > 1 + TINY) || (l0 < 0 - TINY)) err = E_TLOC;
        if (AB) {
            const bool micro = fabs(is.h) <= hmin, full = fabs(is.h - hfull) <= 1e-9 * fabs(hfull);
            multi = micro || (full && p.nhist >= order - 1);
        }
        /* only RK4 steps read the field at their end */
        if (!(AB && multi) && ((l1 > 1 + TINY) || (l1 < 0 - TINY))) err = E_TLOC;
        return true;
    };
    /* the increment of a step that is not RK4 */
    auto multi_inc = [&](double inc[3]) {
        const double h = is.h;
        for (int k = 0; k < 3; k++) {
            const double v = (double)f0[k];
            if (fabs(h) <= hmin) inc[k] = h * v;
            else if (order == 2) inc[k] = h * (3 * v - p.F1[k]) / 2;
            else inc[k] = h * (23 * v - 16 * p.F1[k] + 5 * p.F2[k]) / 12;
        }
    };
    if (!AB) anchor();
    float r = 0.f, s = 0.f, t = 0.f;
    int e = q0, ftag = -1, vtag = -1;
    int4 nd = make_int4(0, 0, 0, 0);
    if (!begin_step() || err) phase = PH_DONE;
    while (phase != PH_DONE) {
        /* ---- one containment test of this lane's walk */
        if (e != ftag) {
            nd = ld32(m.conn, e);
            const Frame F = ld_frame<DIM>(m, e);
            rows[0] = F.a0;
            rows[64] = F.a1;
            if (DIM == 3) rows[128] = F.a2;
            rows[64 * (R::FRAME - 1)] = F.a3;
            ftag = e;
        }
        reload_rows();
        int slot = -1, dec;
        float ge;
        {
            Frame F;
            F.a0 = rows[0];
            F.a1 = rows[64];
            F.a2 = DIM == 3 ? rows[128] : make_float4(0.f, 0.f, 0.f, 0.f);
            F.a3 = rows[64 * (R::FRAME - 1)];
            if (AB && (phase == PH_F0 || phase == PH_LOC)) {
                const float qx = (float)((p.X[0] - m.centre[0]) - (double)F.a0.w);
                const float qy = (float)((p.X[1] - m.centre[1]) - (double)F.a1.w);
                const float qz = DIM == 3 ? (float)((p.X[2] - m.centre[2]) - (double)F.a2.w) : 0.0f;
                frame_nat<DIM>(F, qx, qy, qz, r, s, t);
                ge = F.a3.w;
                gc = 0.0f;
            } else {
                nat_frame<DIM>(F, A, c, r, s, t, ge);
            }
        }
        dec = decide_fast<DIM>(r, s, t, ge, gc, slot);
        if (dec == 2) {
            double x = p.X[0], y = p.X[1], z = p.X[2];
            if (phase != PH_F0 && phase != PH_LOC) {
                x = (m.centre[0] + (double)A[0]) + (double)c[0];
                y = (m.centre[1] + (double)A[1]) + (double)c[1];
                z = (m.centre[2] + (double)A[2]) + (double)c[2];
            }
            const ExactDec xd =
                decide_exact_at<DIM>(m.X64, m.conn, e, x, y, z, phase == PH_LOC ? ACC_SEARCH : ACC_INTERP);
            r = xd.r;
            s = xd.s;
            t = xd.t;
            slot = xd.slot;
            dec = xd.dec;
            tie = tie || xd.tie;
        }
        if (dec < 0) {
            err = E_INDET;
            break;
        }
        if (dec == 0) { /* across the face */
            e = ld32(reinterpret_cast<const int *>(m.adj), 4 * (uint32_t)e + slot);
            if (e != -1) {
                if (++hops >= m.walk_limit) {
                    err = E_WALK;
                    break;
                }
                continue; /* the next test of this walk */
            }
        }
        /* ---- the walk ended: accepted at e, or left the mesh (e == -1) */
        const bool want = e >= 0;
        hops = 0;
        if (phase == PH_LOC) {
            const int start = p.elem;
            p.elem = e;
            if (!want || gone) { /* exit: back to the step's start (integration.c:430-440) */
                const double h6 = is.h * (1.0 / 6.0);
                double inc[3];
                if (AB && multi) multi_inc(inc);
                else
                    for (int k = 0; k < 3; k++) inc[k] = h6 * (double)S[k];
                p.left = 1;
                p.left_time = is.tc - is.h;
                for (int k = 0; k < 3; k++) p.X[k] = p.X[k] - inc[k];
                stop = p.left_time;
                break;
            }
            if (AB) {
                if (!(fabs(is.h) <= hmin)) {
                    if (fabs(is.h - hfull) <= 1e-9 * fabs(hfull)) {
                        for (int k = 0; k < 3; k++) {
                            p.F2[k] = p.F1[k];
                            p.F1[k] = f0[k];
                        }
                        p.nhist = p.nhist < 2 ? p.nhist + 1 : 2;
                    } else {
                        p.nhist = 0;
                    }
                }
                q0 = e; /* the next first stage walks from the located element */
            }
            if (!begin_step() || err) break;
            phase = PH_F0;
            /* the next step's first stage takes this element and these
             * coordinates when the locate started where the first stage
             * started and no test met the tie */
            if (tie || (!AB && start != q0)) {
                e = q0;
                continue;
            }
        }
        gone = gone || !want;
        q0 = q1;
        q1 = q2;
        q2 = q3;
        q3 = e;
        /* ---- this stage's velocity (zero where the probe left, velocity.c:588-592) and the next phase */
        float k[3] = {0.f, 0.f, 0.f};
        if (want) {
            NodeVel<MODE, DIM> g;
            if (e != vtag) {
                gather_vel<MODE, DIM>(f, nd, g);
                vel_to_rows<MODE, DIM>(g, rows + 64 * R::FRAME);
                vtag = e;
            }
            reload_rows();
            vel_from_rows<MODE, DIM>(rows + 64 * R::FRAME, g);
            interp_gathered<MODE, DIM>(f, g, phase == PH_F0 ? tl0 : phase == PH_K4 ? tl1 : tlh, r, s, t, k);
        }
        if (AB && phase == PH_F0) {
            for (int k3 = 0; k3 < 3; k3++) f0[k3] = k[k3];
            if (!multi) {
                anchor();
            } else { /* on to the locate walk, the ring back at the first stage */
                const int last = q3;
                q3 = q2;
                q2 = q1;
                q1 = q0;
                q0 = last;
                phase = PH_K4;
            }
        }
        if (phase == PH_K4) { /* the step's increment, position and time */
            const double h = is.h, h6 = h * (1.0 / 6.0);
            double inc[3];
            if (AB && multi) {
                multi_inc(inc);
            } else {
                for (int k3 = 0; k3 < 3; k3++) {
                    S[k3] = S[k3] + k[k3];
                    inc[k3] = h6 * (double)S[k3];
                }
            }
            for (int k3 = 0; k3 < 3; k3++) p.X[k3] = p.X[k3] + inc[k3];
            is.tc = is.tc + h;
            if (!(fabs(h) <= hmin)) nsteps++;
            taken++;
            if (!AB) anchor();
            tie = false;
            e = p.elem; /* a located element: the walks above keep p.elem >= 0 */
        } else {
            const float hf = (float)is.h, w = phase == PH_K3 ? hf : 0.5f * hf;
            const bool first = phase == PH_F0;
            for (int k3 = 0; k3 < 3; k3++) {
                S[k3] = first ? k[k3] : S[k3] + 2.0f * k[k3];
                c[k3] = D[k3] + w * k[k3];
            }
            gc = guard_offset(m, c);
            e = q0;
        }
        phase++;
    }
    if (err) stop = b;
    if (!ret) { /* suspended at a step's start */
        is.mp[0].elem = q0;
        is.mp[1].elem = q1;
        is.mp[2].elem = q2;
        is.mp[3].elem = q3;
        for (int q = 0; q < 4; q++) is.mp[q].left = 0;
    }
    return ret;
}

/* ------------------------------------------------------------------------ */
/* FP64 RK4 on unstructured meshes, the same state machine                   */
/* ------------------------------------------------------------------------ */
/* The query-independent part of an element's natural coordinates
 * (nat3_exact_p, nat2_exact_p): node 0, the cofactors and the determinant, by
 * the same expressions, with the determinant's inverse for fvc_div_near. */
template <int DIM>
struct Geo64 {
    double x0[DIM], c[DIM][DIM], det, y;
};

template <int DIM>
__device__ __forceinline__ void geo64(const DevMesh &m, int4 nd, Geo64<DIM> &g) {
#pragma clang fp contract(off)
    const double4 p0 = ld32(m.X64, nd.x), p1 = ld32(m.X64, nd.y), p2 = ld32(m.X64, nd.z);
    const double x0 = p0.x, y0 = p0.y, x1 = p1.x, y1 = p1.y, x2 = p2.x, y2 = p2.y;
    g.x0[0] = x0;
    g.x0[1] = y0;
    if constexpr (DIM == 3) {
        const double4 p3 = ld32(m.X64, nd.w);
        const double z0 = p0.z, z1 = p1.z, z2 = p2.z, x3 = p3.x, y3 = p3.y, z3 = p3.z;
        g.x0[2] = z0;
        g.c[0][0] = (z3 - z0) * (y2 - y3) - (z2 - z3) * (y3 - y0);
        g.c[1][0] = (z3 - z0) * (y0 - y1) - (z0 - z1) * (y3 - y0);
        g.c[2][0] = (z1 - z2) * (y0 - y1) - (z0 - z1) * (y1 - y2);
        g.c[0][1] = (x3 - x0) * (z2 - z3) - (x2 - x3) * (z3 - z0);
        g.c[1][1] = (x3 - x0) * (z0 - z1) - (x0 - x1) * (z3 - z0);
        g.c[2][1] = (x1 - x2) * (z0 - z1) - (x0 - x1) * (z1 - z2);
        g.c[0][2] = (y3 - y0) * (x2 - x3) - (y2 - y3) * (x3 - x0);
        g.c[1][2] = (y3 - y0) * (x0 - x1) - (y0 - y1) * (x3 - x0);
        g.c[2][2] = (y1 - y2) * (x0 - x1) - (y0 - y1) * (x1 - x2);
        g.det = (x1 - x0) * ((y2 - y0) * (z3 - z0) - (z2 - z0) * (y3 - y0)) +
                (x2 - x0) * ((y0 - y1) * (z3 - z0) - (z0 - z1) * (y3 - y0)) +
                (x3 - x0) * ((y1 - y0) * (z2 - z0) - (z1 - z0) * (y2 - y0));
    } else {
        g.c[0][0] = y2 - y0;
        g.c[0][1] = x0 - x2;
        g.c[1][0] = y0 - y1;
        g.c[1][1] = x1 - x0;
        g.det = (x1 - x0) * (y2 - y0) - (x2 - x0) * (y1 - y0);
    }
    g.y = fvc_near_inverse(g.det);
}

/* natural coordinates n[0 .. DIM-1] of the point Q */
template <int DIM>
__device__ __forceinline__ void geo64_nat(const Geo64<DIM> &g, const double Q[3], double n[3]) {
#pragma clang fp contract(off)
    double d[DIM], big = 0.0;
    for (int a = 0; a < DIM; a++) d[a] = Q[a] - g.x0[a];
    for (int a = 0; a < DIM; a++) {
        n[a] = g.c[a][0] * d[0] + g.c[a][1] * d[1];
        if (DIM == 3) n[a] = n[a] + g.c[a][2] * d[DIM - 1];
        big = fmax(big, fabs(n[a]));
    }
    if (g.y != 0.0 && big < 1e280)
        for (int a = 0; a < DIM; a++) n[a] = fvc_div_near(n[a], g.det, g.y);
    else
        for (int a = 0; a < DIM; a++) n[a] = n[a] / g.det;
}

/* rk4_sm in FP64 with the reference's expressions (integration.c:317-462):
 * bit for bit the straight-line walks of interval_run.  A lane keeps the
 * geometry of the element it tested last in registers (14 FP64 values in 3-D,
 * with its connectivity and adjacency) and the node velocities of the element
 * it interpolated in last in LDS (192 bytes): a test is then 3 subtractions,
 * 15 multiply-adds and three quotients by one determinant, where the straight
 * walks gathered 144 bytes and ran some 90 operations and three divisions for
 * every test, in five inlined copies.  3 waves per SIMD by both the registers
 * and the LDS (12 KB a wave).  200,003 points in random order in 1.7M tets, 20
 * steps: 2,542 -> 437 us; now bound by the latency of a new element's chain
 * (connectivity, nodes, their velocities), so the adjacency row comes with the
 * connectivity. */
template <int DIM>
__device__ int rk4_sm64(const DevMesh &m, const DevField &f, PState &p, IState &is, double a, double b, double dt,
                        int max_steps, int &err, uint32_t &nsteps, double &stop, float4 *rows) {
#pragma clang fp contract(off)
    constexpr int NN = DIM + 1;
    if (!is.started) {
        if (p.left) {
            err = E_LEFT;
            stop = b;
            return 1;
        }
        if (p.elem < 0 || p.elem >= m.ne) {
            err = E_ELEM;
            stop = b;
            return 1;
        }
        is.tc = a;
        is.h = sign_of(dt, b - a);
        for (int q = 0; q < 4; q++) {
            is.mp[q].elem = p.elem;
            is.mp[q].left = 0;
        }
        is.started = 1;
    }
    const double hmin = 1e-12 * fabs(dt), tinv = fvc_near_inverse(f.tmax - f.tmin);
    int taken = 0, ret = 1;
    int phase = PH_F0, hops = 0, tie = 0;
    bool gone = false;
    int q0 = is.mp[0].elem, q1 = is.mp[1].elem, q2 = is.mp[2].elem, q3 = is.mp[3].elem; /* the ring of rk4_sm */
    double Q[3], S[3] = {0.0, 0.0, 0.0}; /* query point; weighted slope sum */
    double tlh = 0.0, tl1 = 0.0, tl0 = 0.0;
    auto begin_step = [&]() -> bool {
        if (!((is.tc - b) * (b - a) < 0.0)) {
            stop = b;
            return false;
        }
        if (taken == max_steps) {
            ret = 0;
            return false;
        }
        if ((is.tc + is.h - b) * (is.tc + is.h - a) > 0.0) is.h = sign_of(b - is.tc, b - a);
        tl0 = time_loc(f, is.tc, tinv);
        tlh = time_loc(f, is.tc + is.h / 2, tinv); /* lies between tl0 and tl1 */
        tl1 = time_loc(f, is.tc + is.h, tinv);
        if ((tl0 > 1 + TINY) || (tl0 < 0 - TINY) || (tl1 > 1 + TINY) || (tl1 < 0 - TINY)) err = E_TLOC;
        return true;
    };
    for (int c = 0; c < 3; c++) Q[c] = p.X[c];
    int e = q0, gtag = -1, vtag = -1;
    int4 nd = make_int4(0, 0, 0, 0), ad = nd;
    Geo64<DIM> g;
    if (!begin_step() || err) phase = PH_DONE;
    while (phase != PH_DONE) {
        if (e != gtag) {
            nd = ld32(m.conn, e);
            ad = ld32(m.adj, e);
            geo64<DIM>(m, nd, g);
            gtag = e;
        }
        double n[3] = {0.0, 0.0, 0.0};
        geo64_nat<DIM>(g, Q, n);
        int slot = -1;
        const int dec = decide_exact<DIM>(n[0], n[1], n[2], phase == PH_LOC ? ACC_SEARCH : ACC_INTERP, slot, &tie);
        if (dec < 0) {
            err = E_INDET;
            break;
        }
        if (dec == 0) { /* across the face */
            e = slot == 0 ? ad.x : slot == 1 ? ad.y : slot == 2 ? ad.z : ad.w;
            if (e != -1) {
                if (++hops >= m.walk_limit) {
                    err = E_WALK;
                    break;
                }
                continue;
            }
        }
        const bool want = e >= 0;
        hops = 0;
        if (phase == PH_LOC) {
            const int start = p.elem;
            p.elem = e;
            if (!want || gone) { /* exit: back to the step's start (integration.c:430-440) */
                double inc[3];
                for (int c = 0; c < 3; c++) inc[c] = is.h * S[c];
                sixths(inc);
                p.left = 1;
                p.left_time = is.tc - is.h;
                for (int c = 0; c < 3; c++) p.X[c] = p.X[c] - inc[c];
                stop = p.left_time;
                break;
            }
            if (!begin_step() || err) break;
            phase = PH_F0;
            if (tie || start != q0) { /* the first stage walks (see interval_run's reuse) */
                e = q0;
                continue;
            }
        }
        gone = gone || !want;
        q0 = q1;
        q1 = q2;
        q2 = q3;
        q3 = e;
        double k[3] = {0.0, 0.0, 0.0};
        if (want) {
            double2 *vr = reinterpret_cast<double2 *>(rows);
            if (e != vtag) {
                const int ids[4] = {nd.x, nd.y, nd.z, nd.w};
                for (int q = 0; q < NN; q++) {
                    const double4 lo = ld32(reinterpret_cast<const double4 *>(f.lo), ids[q]);
                    const double4 hi = ld32(reinterpret_cast<const double4 *>(f.hi), ids[q]);
                    if constexpr (DIM == 3) {
                        vr[64 * (3 * q)] = make_double2(lo.x, lo.y);
                        vr[64 * (3 * q + 1)] = make_double2(lo.z, hi.x);
                        vr[64 * (3 * q + 2)] = make_double2(hi.y, hi.z);
                    } else {
                        vr[64 * (2 * q)] = make_double2(lo.x, lo.y);
                        vr[64 * (2 * q + 1)] = make_double2(hi.x, hi.y);
                    }
                }
                vtag = e;
            }
            reload_rows();
            /* velocity.c:603-619 */
            const double tl = phase == PH_F0 ? tl0 : phase == PH_K4 ? tl1 : tlh;
            double n0[3];
            for (int q = 0; q < NN; q++) {
                double lo[3], hi[3];
                const double2 u = vr[64 * (DIM * q)], v = vr[64 * (DIM * q + 1)];
                lo[0] = u.x;
                lo[1] = u.y;
                if constexpr (DIM == 3) {
                    const double2 w = vr[64 * (3 * q + 2)];
                    lo[2] = v.x;
                    hi[0] = v.y;
                    hi[1] = w.x;
                    hi[2] = w.y;
                } else {
                    hi[0] = v.x;
                    hi[1] = v.y;
                }
                for (int c = 0; c < DIM; c++) {
                    const double at = (1 - tl) * lo[c] + tl * hi[c];
                    if (q == 0) k[c] = n0[c] = at;
                    else k[c] = k[c] + (at - n0[c]) * fabs(n[q - 1]);
                }
            }
        }
        if (phase == PH_K4) {
            double inc[3];
            for (int c = 0; c < 3; c++) {
                S[c] = S[c] + k[c];
                inc[c] = is.h * S[c];
            }
            sixths(inc);
            for (int c = 0; c < 3; c++) Q[c] = p.X[c] = p.X[c] + inc[c];
            if (!(fabs(is.h) <= hmin)) nsteps++;
            is.tc = is.tc + is.h;
            taken++;
            tie = 0;
            e = p.elem;
        } else {
            const bool first = phase == PH_F0;
            const double w = phase == PH_K3 ? 1.0 : 0.5;
            for (int c = 0; c < 3; c++) {
                S[c] = first ? k[c] : S[c] + 2 * k[c];
                Q[c] = p.X[c] + w * k[c] * is.h;
            }
            e = q0;
        }
        phase++;
    }
    if (err) stop = b;
    if (!ret) { /* suspended at a step's start */
        is.mp[0].elem = q0;
        is.mp[1].elem = q1;
        is.mp[2].elem = q2;
        is.mp[3].elem = q3;
        for (int q = 0; q < 4; q++) is.mp[q].left = 0;
    }
    return ret;
}

/* RK4 on a Cartesian grid (integration.c:317-462) without strain rate or
 * extrapolation.  One copy of the stage's interpolation in a loop over the
 * four stages, with the weighted slope sum built as they come, in the
 * reference's order: four copies side by side hold all four slopes and spill
 * (the FP64 3-D kernel 80 registers).  What bounds the FP64 kernel is its
 * chain of dependent instructions: about 180 a stage, 490 with the divisions
 * and the zero-weight corners.  512x256 FTLE points of the double gyre, 50
 * steps: 499 us; without those divisions and corners 264 us; with the axes'
 * quotients side by side and the cell's corners in LDS 209 us. */
template <int MODE, int DIM>
__device__ int rk4_cart(const DevMesh &m, const DevField &f, PState &p, IState &is, double a, double b, double dt,
                        int max_steps, int &err, uint32_t &nsteps, double &stop, float4 *rows) {
#pragma clang fp contract(off)
    if (!is.started) {
        if (p.left) {
            err = E_LEFT;
            stop = b;
            return 1;
        }
        is.tc = a;
        is.h = sign_of(dt, b - a);
        is.started = 1;
    }
    const double hmin = 1e-12 * fabs(dt), tinv = fvc_near_inverse(f.tmax - f.tmin);
    CartLast last;
    last.rows = rows;
    int taken = 0;
    stop = b;
    while ((is.tc - b) * (b - a) < 0.0) {
        if (taken == max_steps) return 0;
        if ((is.tc + is.h - b) * (is.tc + is.h - a) > 0.0) is.h = sign_of(b - is.tc, b - a);
        const double h = is.h;
        double Y[3], S[3] = {0.0, 0.0, 0.0};
        bool out = false;
        for (int c = 0; c < 3; c++) Y[c] = p.X[c];
#pragma unroll 1
        for (int stage = 0; stage < 4; stage++) {
            const double tq = stage == 0 ? is.tc : stage == 3 ? is.tc + h : is.tc + h / 2;
            double k[3] = {0.0, 0.0, 0.0}, loc[3];
            int cell[3];
            if (cart_cell<DIM>(m, Y, cell, loc)) {
                const double tloc = time_loc(f, tq, tinv);
                if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
                    err = E_TLOC;
                    break;
                }
                cart_velocity<MODE, DIM>(m, f, tloc, cell, loc, last, k);
            } else {
                out = true; /* zero velocity for this stage */
            }
            const double w = stage == 2 ? 1.0 : 0.5, u = stage == 3 ? 1.0 : 2.0;
            for (int c = 0; c < 3; c++) {
                S[c] = stage == 0 ? k[c] : S[c] + u * k[c];
                Y[c] = p.X[c] + w * k[c] * h;
            }
        }
        if (err) return 1;
        double inc[3];
        for (int c = 0; c < 3; c++) inc[c] = h * S[c];
        sixths(inc);
        for (int c = 0; c < 3; c++) p.X[c] = p.X[c] + inc[c];
        is.tc = is.tc + h;
        if (!(fabs(h) <= hmin)) nsteps++;
        taken++;
        if (out || outside_domain(m, p.X[0], p.X[1], p.X[2])) {
            p.left = 1;
            p.left_time = is.tc - h;
            for (int c = 0; c < 3; c++) p.X[c] = p.X[c] - inc[c];
            stop = p.left_time;
            return 1;
        }
    }
    return 1;
}

/* Returns 1 when the interval is finished (end reached, point exited or an
 * error), with *stop the stop time; 0 when max_steps were taken first.
 *   RK4   ompVC/integration.c:317-462
 *   Euler ompVC/integration.c:222-311 (GetVelocity on the point itself)
 *   AB2/AB3 (no ompVC counterpart; cudaVC/src/multistep.cu:249-304 is not
 *   followed): x+ = x + h (3 f0 - f1)/2, x+ = x + h (23 f0 - 16 f1 + 5 f2)/12
 *   with f0 = u(x, t); RK4 steps while the history is short or the step is
 *   clipped by more than 1e-9 h (history restarts); steps below 1e-12 dt
 *   (accumulation remainders) are Euler steps that keep the history. */
template <int MODE, int DIM, int UNSTRUCT, int GEN>
__device__ int interval_run(const DevMesh &m, const DevField &f, PState &p, IState &is, double a, double b, double dt,
                            int itype_rt, int extrap, int max_steps, int &err, uint32_t &nsteps, double &stop,
                            float4 *rows = nullptr) {
#pragma clang fp contract(off)
    /* GEN = 0 and 3 compile RK4 only (no multistep state in registers) */
    const int itype = GEN == 0 || GEN == 3 ? INT_RK4 : itype_rt;
    if constexpr (MODE == P_F64 && UNSTRUCT && !GEN) {
        if (!extrap) return rk4_sm64<DIM>(m, f, p, is, a, b, dt, max_steps, err, nsteps, stop, rows);
    }
    if constexpr (MODE != P_F64 && UNSTRUCT && GEN == 2) { /* AB2 and AB3 without strain rate, exposure time, extrapolation */
        return rk4_sm<MODE, DIM, 1>(m, f, p, is, a, b, dt, max_steps, err, nsteps, stop, rows, itype_rt);
    }
    if constexpr (MODE != P_F64 && UNSTRUCT && !GEN) {
        /* GEN = 0 builds integrate RK4 only, without strain rate or exposure
         * time; the GEN = 1 builds (other integrators, RK4 with extrapolation
         * or those integrals) keep the straight-line walks below and leave
         * the state machine's registers out */
        if (!extrap) return rk4_sm<MODE, DIM>(m, f, p, is, a, b, dt, max_steps, err, nsteps, stop, rows);
    }
    if constexpr (!UNSTRUCT && !GEN) {
        if (!extrap) return rk4_cart<MODE, DIM>(m, f, p, is, a, b, dt, max_steps, err, nsteps, stop, rows);
    }
    if (!is.started) {
        if (p.left) {
            err = E_LEFT;
            stop = b;
            return 1;
        }
        if (UNSTRUCT && (p.elem < 0 || p.elem >= m.ne)) {
            err = E_ELEM;
            stop = b;
            return 1;
        }
        is.tc = a;
        is.h = sign_of(dt, b - a);
        for (int q = 0; q < 4; q++) {
            is.mp[q].elem = p.elem;
            is.mp[q].left = 0;
        }
        is.started = 1;
    }
    const double hfull = sign_of(dt, b - a);
    const double hmin = 1e-12 * fabs(dt);
    const int order = itype == INT_AB2 ? 2 : 3;
    int taken = 0;
    /* The locate walk at the end of a step starts from the point's element
     * and seeks the new position; the next step's first-stage walk seeks the
     * same position from the first probe's element.  When the two start
     * elements are equal (the usual case: both hold the previous position)
     * the walks visit the same elements and take the same decisions (the
     * acceptance rules d > -TINY and d + TINY >= 0 differ only at
     * d == -TINY, which voids the reuse), so the first stage takes the
     * locate's element and natural coordinates without walking again. */
    int c_elem = -1;
    /* activation potential (integration.c:355-360, 449-455): Scalar gains
     * h (S0 + S1) / 2 per step that stays in the domain, S0 and S1 the strain
     * rate at the step's start and end; only the generic integrator build */
    const bool ap = GEN == 1 && f.sr_lo != nullptr;
    const bool cet = GEN == 1 && UNSTRUCT && f.cet_lo != nullptr; /* exposure time (integration.c:427-448) */
    using CT = typename VelT<MODE>::T; /* reduced-precision interpolation reads (float) r, s, t */
    CT c_r = 0, c_s = 0, c_t = 0;
    /* Reduced-precision modes on unstructured meshes integrate in FP32: stage
     * velocities, probes (relative to the mesh centre) and the weighted sum
     * of the four slopes; the position and time stay FP64, the increment is
     * h times the FP32 slope sum over 6 in FP64. */
    constexpr bool FAST = MODE != P_F64 && UNSTRUCT;
    using KT = typename std::conditional<FAST, float, double>::type;
    /* FAST: time locations as (t - tmin) times one reciprocal of the frame span */
    const double inv_span = FAST ? 1.0 / (f.tmax - f.tmin) : 0.0;
    const double tinv = FAST ? 0.0 : fvc_near_inverse(f.tmax - f.tmin);
    CartLast last;
    if (!UNSTRUCT && !GEN) last.rows = rows;
    while ((is.tc - b) * (b - a) < 0.0) {
        if (taken == max_steps) return 0;
        if ((is.tc + is.h - b) * (is.tc + is.h - a) > 0.0) is.h = sign_of(b - is.tc, b - a);
        const double h = is.h, tc = is.tc;
        const bool micro = fabs(h) <= hmin;
        double inc[3], sr0 = 0.0;
        KT f0[3];
        if (ap) {
            sr0 = strain_rate<DIM, UNSTRUCT>(m, f, tc, p, err);
            if (err) break;
        }
        bool ab_step = false;
        if (itype == INT_EULER) {
            double ve[3];
            get_velocity<MODE, DIM>(m, f, tc, p, ve, err);
            if (err) break;
            for (int c = 0; c < 3; c++) inc[c] = h * ve[c];
        } else {
            if (UNSTRUCT && c_elem >= 0) {
                const double tloc = FAST ? (tc - f.tmin) * inv_span : time_loc(f, tc, tinv);
                if ((tloc > 1 + TINY) || (tloc < 0 - TINY)) {
                    err = E_TLOC;
                    break;
                }
                is.mp[0].elem = c_elem;
                if constexpr (FAST) interp_unstruct_f<MODE, DIM>(m, f, (float)tloc, c_elem, c_r, c_s, c_t, f0);
                else interp_unstruct<MODE, DIM>(m, f, tloc, c_elem, c_r, c_s, c_t, f0);
            } else {
                if constexpr (FAST) stage_velocity_x<MODE, DIM>(m, f, (tc - f.tmin) * inv_span, p.X, is.mp[0], f0, err);
                else stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc, p.X, is.mp[0], f0, err, tinv, last);
            }
            c_elem = -1;
            if (err) break;
            const bool full = fabs(h - hfull) <= 1e-9 * fabs(hfull);
            if (itype != INT_RK4 && micro) {
                for (int c = 0; c < 3; c++) inc[c] = h * (double)f0[c];
            } else if (itype != INT_RK4 && full && p.nhist >= order - 1) {
                ab_step = true;
                if (order == 2)
                    for (int c = 0; c < 3; c++) inc[c] = h * (3 * (double)f0[c] - p.F1[c]) / 2;
                else
                    for (int c = 0; c < 3; c++)
                        inc[c] = h * (23 * (double)f0[c] - 16 * p.F1[c] + 5 * p.F2[c]) / 12;
            } else if constexpr (FAST) {
                /* k2, k3, k4 at probes X + h/2 f0, X + h/2 k2, X + h k3 (anchor A,
                 * offset D + c h k); S = f0 + 2 k2 + 2 k3 + k4 */
                const float hf = (float)h, hh = 0.5f * hf;
                const double tl_half = (tc + h / 2 - f.tmin) * inv_span, tl_end = (tc + h - f.tmin) * inv_span;
                float A[3], D[3], d[3], k[3], S[3];
                for (int c = 0; c < 3; c++) {
                    const double xc = p.X[c] - m.centre[c];
                    A[c] = (float)xc;
                    D[c] = (float)(xc - (double)A[c]);
                    S[c] = f0[c];
                    d[c] = D[c] + hh * f0[c];
                }
                stage_velocity_c<MODE, DIM>(m, f, tl_half, A, d, is.mp[1], k, err);
                if (err) break;
                for (int c = 0; c < 3; c++) {
                    S[c] = S[c] + 2.0f * k[c];
                    d[c] = D[c] + hh * k[c];
                }
                stage_velocity_c<MODE, DIM>(m, f, tl_half, A, d, is.mp[2], k, err);
                if (err) break;
                for (int c = 0; c < 3; c++) {
                    S[c] = S[c] + 2.0f * k[c];
                    d[c] = D[c] + hf * k[c];
                }
                stage_velocity_c<MODE, DIM>(m, f, tl_end, A, d, is.mp[3], k, err);
                if (err) break;
                const double h6 = h * (1.0 / 6.0);
                for (int c = 0; c < 3; c++) inc[c] = h6 * (double)(S[c] + k[c]);
            } else {
                double k2[3], k3[3], k4[3], Y[3];
                for (int c = 0; c < 3; c++) Y[c] = p.X[c] + 0.5 * f0[c] * h;
                stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + h / 2, Y, is.mp[1], k2, err, tinv, last);
                if (err) break;
                for (int c = 0; c < 3; c++) Y[c] = p.X[c] + 0.5 * k2[c] * h;
                stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + h / 2, Y, is.mp[2], k3, err, tinv, last);
                if (err) break;
                for (int c = 0; c < 3; c++) Y[c] = p.X[c] + k3[c] * h;
                stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + h, Y, is.mp[3], k4, err, tinv, last);
                if (err) break;
                for (int c = 0; c < 3; c++) inc[c] = h * (f0[c] + 2 * k2[c] + 2 * k3[c] + k4[c]);
                sixths(inc);
            }
            (void)ab_step;
        }
        for (int c = 0; c < 3; c++) p.X[c] = p.X[c] + inc[c];
        is.tc = tc + h;
        if (!micro) nsteps++;
        taken++;
        bool out;
        if (UNSTRUCT) {
            double r, s, t;
            const int start = p.elem;
            int tie = 0;
            int e = p.elem < 0 ? -1
                               : walk<MODE, DIM>(m, p.X[0], p.X[1], p.X[2], p.elem, ACC_SEARCH, r, s, t, err, &tie);
            if (e == -2) break;
            p.elem = e;
            out = e < 0;
            /* RK4: the next first-stage walk starts at mp[0]; AB: at the located element */
            if (e >= 0 && !tie && itype != INT_EULER && (itype != INT_RK4 || start == is.mp[0].elem)) {
                c_elem = e;
                c_r = (CT)r;
                c_s = (CT)s;
                c_t = (CT)t;
            }
        } else {
            out = outside_domain(m, p.X[0], p.X[1], p.X[2]);
        }
        if (itype != INT_EULER)
            out = out || is.mp[0].left || is.mp[1].left || is.mp[2].left || is.mp[3].left;
        if (out) {
            p.left = 1;
            p.left_time = is.tc - h;
            for (int c = 0; c < 3; c++) p.X[c] = p.X[c] - inc[c];
            stop = p.left_time;
            return 1;
        }
        if (cet) { /* the step's start as the reference recomputes it: X1 minus the increment */
            double X0[3];
            for (int c = 0; c < 3; c++) X0[c] = p.X[c] - inc[c];
            cet_step<DIM>(m, f, X0, p.X, p.elem, h, err);
            if (err) break;
        }
        if (ap) {
            const double sr1 = strain_rate<DIM, UNSTRUCT>(m, f, is.tc, p, err);
            if (err) break;
            p.scalar += (h * ((sr0 + sr1) / 2));
        }
        if (itype == INT_AB2 || itype == INT_AB3) {
            if (!micro) {
                if (fabs(h - hfull) <= 1e-9 * fabs(hfull)) {
                    for (int c = 0; c < 3; c++) {
                        p.F2[c] = p.F1[c];
                        p.F1[c] = f0[c];
                    }
                    p.nhist = p.nhist < 2 ? p.nhist + 1 : 2;
                } else {
                    p.nhist = 0;
                }
            }
            if (UNSTRUCT) is.mp[0].elem = p.elem; /* next f0 walks from the located element */
        }
        if (extrap) {
            get_velocity<MODE, DIM>(m, f, is.tc, p, p.V, err);
            if (err) break;
        }
    }
    stop = b;
    return 1;
}

/* Runge-Kutta-Fehlberg 4(5) over [a, b] (ompVC/integration.c:464-699): the
 * fourth-order result is kept and the step adapted from its difference to
 * the fifth-order one; the step starts at Int_MaxTimeStep every call and six
 * probes keep their own elements within the call.  A probe outside stops the
 * point at the step's start time, without revert; a position outside after
 * an accepted step is reverted as in RK4.  Accepted steps are counted. */
template <int MODE, int DIM, int UNSTRUCT>
__device__ double rkf_run(const DevMesh &m, const DevField &f, PState &p, double a, double b, int extrap, int &err,
                          uint32_t &nsteps) {
#pragma clang fp contract(off)
    if (p.left) {
        err = E_LEFT;
        return b;
    }
    if (UNSTRUCT && (p.elem < 0 || p.elem >= m.ne)) {
        err = E_ELEM;
        return b;
    }
    Probe mp[6];
    for (int q = 0; q < 6; q++) {
        mp[q].elem = p.elem;
        mp[q].left = 0;
    }
    const double a3 = 3.0 / 32.0, b3 = 9.0 / 32.0;
    const double a4 = 1932.0 / 2197.0, b4 = -7200.0 / 2197.0, c4 = 7296.0 / 2197.0;
    const double a5 = 439.0 / 216.0, b5 = -8.0, c5 = 3680.0 / 513.0, d5 = -845.0 / 4104.0;
    const double a6 = -8.0 / 27.0, b6 = 2.0, c6 = -3544.0 / 2565.0, d6 = 1859.0 / 4104.0, e6 = -11.0 / 40.0;
    const double a7 = 1.0 / 360.0, b7 = -128.0 / 4275.0, c7 = -2197.0 / 75240.0, d7 = 1.0 / 50.0, e7 = 2.0 / 55.0;
    const double a8 = 25.0 / 216.0, b8 = 1408.0 / 2565.0, c8 = 2197.0 / 4104.0, d8 = -1.0 / 5.0;
    const double hmax = f.rkf_max, hmin = f.rkf_min, tol = f.rkf_tol;
    const bool ap = f.sr_lo != nullptr;                 /* activation potential (integration.c:534-539, 671-677) */
    const bool cet = UNSTRUCT && f.cet_lo != nullptr;   /* exposure time (integration.c:650-670) */
    const double tinv = fvc_near_inverse(f.tmax - f.tmin);
    CartLast last; /* gathers every time */
    double h = sign_of(hmax, b - a), tc = a;
    double k1[3], k2[3], k3[3], k4[3], k5[3], k6[3], Y[3];
    while ((tc - b) * (b - a) < 0.0) {
        if ((tc + h - b) * (tc + h - a) > 0.0) h = sign_of(b - tc, b - a);
        double sr0 = 0.0;
        if (ap) {
            sr0 = strain_rate<DIM, UNSTRUCT>(m, f, tc, p, err);
            if (err) return b;
        }
        stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc, p.X, mp[0], k1, err, tinv, last);
        if (err) return b;
        for (int c = 0; c < 3; c++) Y[c] = p.X[c] + 0.25 * k1[c] * h;
        stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + 0.25 * h, Y, mp[1], k2, err, tinv, last);
        if (err) return b;
        for (int c = 0; c < 3; c++) Y[c] = p.X[c] + (a3 * k1[c] + b3 * k2[c]) * h;
        stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + 0.375 * h, Y, mp[2], k3, err, tinv, last);
        if (err) return b;
        for (int c = 0; c < 3; c++) Y[c] = p.X[c] + (a4 * k1[c] + b4 * k2[c] + c4 * k3[c]) * h;
        stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + (12.0 * h) / 13.0, Y, mp[3], k4, err, tinv, last);
        if (err) return b;
        for (int c = 0; c < 3; c++) Y[c] = p.X[c] + (a5 * k1[c] + b5 * k2[c] + c5 * k3[c] + d5 * k4[c]) * h;
        stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + h, Y, mp[4], k5, err, tinv, last);
        if (err) return b;
        for (int c = 0; c < 3; c++)
            Y[c] = p.X[c] + (a6 * k1[c] + b6 * k2[c] + c6 * k3[c] + d6 * k4[c] + e6 * k5[c]) * h;
        stage_velocity<MODE, DIM, UNSTRUCT>(m, f, tc + 0.5 * h, Y, mp[5], k6, err, tinv, last);
        if (err) return b;
        if (mp[0].left || mp[1].left || mp[2].left || mp[3].left || mp[4].left || mp[5].left) {
            p.left = 1;
            p.left_time = tc;
            return tc;
        }
        double er = 0.0;
        for (int c = 0; c < 3; c++) {
            const double ec = fabs(a7 * k1[c] + b7 * k3[c] + c7 * k4[c] + d7 * k5[c] + e7 * k6[c]);
            er = c == 0 ? ec : fmax(er, ec);
        }
        double ss = er == 0.0 ? 0.0 : fvc_root4_rn(fabs((tol * h) / (2 * er)));
        if (er < tol || fabs(h) <= hmin) {
            double inc[3];
            for (int c = 0; c < 3; c++) {
                inc[c] = (a8 * k1[c] + b8 * k3[c] + c8 * k4[c] + d8 * k5[c]) * h;
                p.X[c] = p.X[c] + inc[c];
            }
            tc = tc + h;
            nsteps++;
            bool out;
            if (UNSTRUCT) {
                double r, s, t;
                const int e = walk<MODE, DIM>(m, p.X[0], p.X[1], p.X[2], p.elem, ACC_SEARCH, r, s, t, err);
                if (e == -2) return b;
                p.elem = e;
                out = e < 0;
            } else {
                out = outside_domain(m, p.X[0], p.X[1], p.X[2]);
            }
            if (out) {
                p.left = 1;
                p.left_time = tc - h;
                for (int c = 0; c < 3; c++) p.X[c] = p.X[c] - inc[c];
                return p.left_time;
            }
            if (extrap) {
                get_velocity<MODE, DIM>(m, f, tc, p, p.V, err);
                if (err) return b;
            }
            if (cet) {
                double X0[3];
                for (int c = 0; c < 3; c++) X0[c] = p.X[c] - inc[c];
                cet_step<DIM>(m, f, X0, p.X, p.elem, h, err);
                if (err) return b;
            }
            if (ap) {
                const double sr1 = strain_rate<DIM, UNSTRUCT>(m, f, tc, p, err);
                if (err) return b;
                p.scalar += (h * ((sr0 + sr1) / 2));
            }
            if (fabs(h) > hmin && ss > 1.0) {
                ss = ss > 4.0 ? 4.0 : ss;
                h = sign_of(fabs(ss * h) > hmax ? hmax : ss * h, b - a);
            }
        } else if (ss < 1.0) {
            ss = ss < 0.1 ? 0.1 : ss;
            h = sign_of(fabs(ss * h) < hmin ? hmin : ss * h, b - a);
        } else {
            h = sign_of(fabs(0.5 * h) < hmin ? hmin : 0.5 * h, b - a);
        }
    }
    return b;
}

/* Advect (ompVC/integration.c:22-45) over [t1, t2] in one go */
template <int MODE, int DIM, int UNSTRUCT, int GEN = 1>
__device__ __forceinline__ double advect(const DevMesh &m, const DevField &f, PState &p, double t1, double t2, int itype,
                                         double dt, int extrap, int &err, uint32_t &nsteps, float4 *rows = nullptr) {
#pragma clang fp contract(off)
    if (p.left && extrap) {
        for (int c = 0; c < 3; c++) p.X[c] = p.X[c] + p.V[c] * (t2 - t1);
        return t2;
    }
    double stop = t2;
    if (GEN == 1 && itype == INT_RKF) {
        stop = rkf_run<MODE, DIM, UNSTRUCT>(m, f, p, t1, t2, extrap, err, nsteps);
    } else {
        IState is;
        is.started = 0;
        interval_run<MODE, DIM, UNSTRUCT, GEN>(m, f, p, is, t1, t2, dt, itype, extrap, 0x7fffffff, err, nsteps, stop,
                                               rows);
    }
    if ((fabs(stop - t2) > TINY) && extrap)
        for (int c = 0; c < 3; c++) p.X[c] = p.X[c] + p.V[c] * (t2 - stop);
    return stop;
}


/* ------------------------------------------------------------------------ */
/* largest eigenvalue of a symmetric 3x3, cyclic Jacobi rotations (FP64)     */
/* (Golub & Van Loan, Matrix Computations, sec. 8.5)                          */
/* ------------------------------------------------------------------------ */
__device__ __forceinline__ double max_eig_sym3(double a[3][3], int &err) {
#pragma clang fp contract(off)
    for (int i = 0; i < 3; i++)
        for (int j = i + 1; j < 3; j++) a[i][j] = a[j][i] = 0.5 * (a[i][j] + a[j][i]);
    for (int sweep = 0; sweep < 64; sweep++) {
        double off = fabs(a[0][1]) + fabs(a[0][2]) + fabs(a[1][2]);
        double diag = fabs(a[0][0]) + fabs(a[1][1]) + fabs(a[2][2]);
        if (off == 0.0 || off <= 1e-300 || off < 1e-18 * diag) break;
        if (sweep == 63) err = E_EIG;
#pragma unroll
        for (int pq = 0; pq < 3; pq++) {
            int p = pq == 2 ? 1 : 0, q = pq == 0 ? 1 : 2;
            double apq = a[p][q];
            if (apq == 0.0) continue;
            double theta = (a[q][q] - a[p][p]) / (2.0 * apq);
            double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
            if (!isfinite(theta) || fabs(theta) > 1e150) t = 0.5 / theta;
            double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
            double app = a[p][p], aqq = a[q][q];
            a[p][p] = app - t * apq;
            a[q][q] = aqq + t * apq;
            a[p][q] = a[q][p] = 0.0;
            int r = 3 - p - q;
            double arp = a[r][p], arq = a[r][q];
            a[r][p] = a[p][r] = c * arp - s * arq;
            a[r][q] = a[q][r] = s * arp + c * arq;
        }
    }
    double m = a[0][0] > a[1][1] ? a[0][0] : a[1][1];
    return m > a[2][2] ? m : a[2][2];
}

} // namespace fvc
