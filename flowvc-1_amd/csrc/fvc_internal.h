/*
 * fvc_internal.h - shared between the C ABI (fvc_api.hip) and the kernel
 * launchers (fvc_kernels.hip).  Not part of the public interface.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <set>
#include <string>
#include <vector>

#include "fvc.h"
#include "fvc_device.h"

/* what the kernels report to the host after a launch */
struct fvc_status {
    /* particle-steps and idle lanes of the advection launches, never cleared
     * (take_steps takes the differences); particle-steps of batches and servers */
    unsigned long long steps[3];
    int64_t where;               /* point of the first error */
    int err;                     /* first error code, 0 if none */
    int count;                   /* length of the last compacted list */
};

struct fvc_ctx {
    int device;
    int precision;
    hipStream_t stream;
    fvc::DevMesh mesh;
    /* device allocations */
    double4 *X64;
    float4 *ER; /* element frames, 4 per element */
    int4 *conn, *adj;
    int *cell_start, *cell_elems;
    int64_t ncells, nentries;
    /* resident velocity slices */
    int max_slices;
    std::vector<void *> slices;
    std::vector<float> slice_scale;
    std::vector<double> slice_time;
    std::vector<int> slice_vals; /* VALS_* of each slice, looked at for 2-D grids in FP64 */
    std::vector<double> slice_speed; /* unstructured meshes: rms speed of each slice, by a sample of its nodes */
    double edge = 0.0;  /* unstructured meshes: mean element edge, by a sample of the elements */
    int64_t nvel;       /* nodes per slice */
    size_t vel_stride;  /* bytes per node */
    /* resident strain-rate slices (activation potential), FP64, one per slot */
    std::vector<double *> sr_slices;
    int64_t nsr; /* values per strain-rate slice: elements, or Cartesian cells */
    /* exposure time: per element 128-bit fixed-point sums (low, high words) and encounters */
    unsigned long long *cet_lo, *cet_hi;
    int *cet_enc;
    /* errors and counters: d_err, d_where and d_steps point into d_status,
     * which check_err copies back whole into the pinned h_status with one
     * copy and one stream synchronisation */
    fvc_status *d_status, *h_status;
    int *d_err;
    int64_t *d_where;
    unsigned long long *d_steps;
    unsigned long long steps_seen[2]; /* steps[0], steps[1] when last taken */
    int64_t last_steps;
    int64_t last_idle; /* lanes of the last fvc_advect or fvc_ftle_frame launch whose particle was not integrated */
    std::string last_error;
    int64_t bytes_used;
    /* scratch (grown on demand) */
    void *scratch;
    size_t scratch_bytes;
    /* pinned ring of outputs (out_chunks), at most 8 MB, with one event per
     * slot; small outputs go through the pinned block that h_status begins,
     * and so does the first one that is not (staged_once) */
    char *stage;
    size_t stage_bytes;
    bool staged_once;
    std::vector<hipEvent_t> stage_ev;
    /* side stream: an FTLE slide frame's early FTLE (from a snapshot of its
     * stencils) runs there beside the next frame's advection; side_done
     * follows the last launch on it, side_pending until the main stream or
     * the host has waited for it */
    hipStream_t side;
    hipEvent_t side_ready, side_done;
    int side_pending;
    /* kernel timing (HIP events on `stream`) */
    int timing;
    int chain_replay; /* seed chains: 1 = always the point-by-point replay */
    hipEvent_t ev0, ev1;
    double t_ms;
    int64_t t_launches, t_steps;
    /* objects created on this context: fvc_destroy releases their device
     * memory and detaches them (their handles then accept only *_destroy) */
    std::set<fvc_particles *> live_particles;
    std::set<fvc_ftle *> live_ftle;
    std::set<fvc_batch *> live_batches;
    std::set<fvc_server *> live_servers;
};

struct fvc_particles {
    fvc_ctx *ctx; /* null once detached by fvc_destroy */
    int64_t cap;
    void *buf;
    double *X[3];
    double *V[3];
    int *elem, *aux, *left;
    double *left_time, *scalar;
    double *H[6]; /* multistep history F1 (x,y,z), F2 (x,y,z) */
    int *nhist;
    /* particles still to integrate in [act_begin, act_begin + act_count), as
     * indices relative to act_begin (built by fvc_advect, dropped by any
     * write of particle state from outside the integrators) */
    int *act = nullptr;
    int64_t act_begin = -1, act_count = 0, act_n = 0;
    int act_extrap = 0;
};

struct fvc_ftle {
    fvc_ctx *ctx; /* null once detached by fvc_destroy */
    double mn[3], mx[3], del[3];
    int32_t res[3];
    int64_t n;
    double start_time, stop_time;
    int status; /* 0 unlaunched, 1 launched, 2 complete */
    fvc_particles *pts;
    /* per point */
    int *have;
    double *wt, *wot;
    /* staging of one frame */
    double *Xn[3];
    int *elem_new;
    int *exited;   /* 1 when the point left during this frame */
    int *advected; /* 1 when the point was integrated this frame */
    double *exit_time;
    double *Vn[3];
    int *active;    /* compacted indices of points to integrate (Z-ordered) */
    int *zperm;     /* grid points in Z-order */
    int64_t nactive;     /* length of `active`, -1: to be built */
    int active_extrap;   /* the extrapolation flag it was built for */
    int64_t active_gone; /* points on it that had left when the last frame began */
    /* stencil snapshots of the early FTLE, used by alternate frames */
    void *snap[2];
    int64_t snap_cap;
    int snap_sel;
    void *buf;
    int64_t inside;
    /* state right after creation, for fvc_ftle_reset */
    fvc_particles *init_pts;
    int *init_have;
    double *init_w;
};

/* launchers (fvc_kernels.hip); all return FVC_OK or a negative code */
namespace fvc {
struct PtrSet {
    double *X[3];
    double *V[3];
    int *elem;
    int *left;
    double *left_time;
    double *H[6];
    int *nhist;
    double *scalar = nullptr; /* LagrangianPoint.Scalar (activation potential) */
};

inline PtrSet ptrs(fvc_particles *p) {
    PtrSet s;
    for (int c = 0; c < 3; c++) {
        s.X[c] = p->X[c];
        s.V[c] = p->V[c];
    }
    for (int c = 0; c < 6; c++) s.H[c] = p->H[c];
    s.elem = p->elem;
    s.left = p->left;
    s.left_time = p->left_time;
    s.nhist = p->nhist;
    return s; /* scalar stays null: only activation-potential runs carry it */
}

/* one FTLE grid's device arrays (grid index P = (i*res1 + j)*res2 + k) */
struct FtleDev {
    int res[3];
    double del[3];
    double start_time;
    PtrSet p;
    int *have;
    double *wt, *wot;
    double *Xn[3], *Vn[3];
    int *elem_new, *exited, *advected;
    double *exit_time;
    int *early_nt = nullptr; /* counter of triggered points that the frame's advection clears */
};
FtleDev ftle_dev(fvc_ftle *f);

DevField bind_field(fvc_ctx *c, int lo, int hi, double tmin, double tmax);

int launch_velocity(fvc_ctx *c, PtrSet p, int64_t begin, int64_t count, double t, const DevField &f);
int launch_cet_encounters(fvc_ctx *c, PtrSet p, int64_t begin, int64_t count, int *enc);
int launch_advect_times(fvc_ctx *c, PtrSet p, int64_t begin, int64_t count, const double *dtt, const DevField &f,
                        const fvc_int_params &ip);
int launch_active_list(fvc_ctx *c, PtrSet p, int64_t begin, int64_t count, int extrap, int *list, int64_t *n);
int launch_advect(fvc_ctx *c, PtrSet p, const int *index, int64_t begin, int64_t count, double t1, double t2,
                  const DevField &f, const fvc_int_params &ip);
int launch_locate(fvc_ctx *c, const double *dxyz, const int *dguess, int64_t n, int mode, int *dout);
/* chain: 0 = point list (ReadInTraceMesh), 1 = tracer grid (GenerateTracerMesh), 2 = FTLE grid */
/* device sorting helpers (any stream) */
int radix_sort_pairs(hipStream_t s, uint64_t *k0, int *v0, uint64_t *k1, int *v1, int64_t n, int bits, int *which);
int scan_exclusive_small(hipStream_t s, int *a, int n);
int launch_seed_chain(fvc_ctx *c, int chain, int64_t n, const double *dxyz, const double mn[3], const double del[3],
                      const int32_t res[3], int lsc, int *d_elem, int *d_left, double *d_left_time);
int launch_ftle_frame(fvc_ftle *f, int lo, int hi, double tmin, double tmax, double t1, double t2,
                      const fvc_int_params &ip);
int launch_ftle_fill(fvc_ftle *f, double int_t);
int launch_ftle_mask(fvc_ftle *f);
/* the same on any FTLE grid view (enqueue only, no synchronisation) */
int launch_ftle_early(fvc_ctx *c, const FtleDev &d, int64_t n, const DevField &fld, double t1, int itype, double dt);
int launch_ftle_update_all(fvc_ctx *c, const FtleDev &d, int64_t n, int extrap);
int launch_ftle_fill_dev(fvc_ctx *c, const FtleDev &d, int64_t n, double int_t);
int launch_ftle_mask_dev(fvc_ctx *c, const FtleDev &d, int64_t n);
/* indices i (or map[i]) of the nonzero flags, in order */
int launch_compact(fvc_ctx *c, const int *flags, int64_t n, int *out_idx, int64_t *count, const int *map = nullptr);
/* Z-order (Morton, i most significant) permutation of the points of a grid */
int launch_grid_zorder(fvc_ctx *c, const int32_t res[3], int64_t n, int *dperm);
int launch_zsort(fvc_ctx *c, const double *dxyz, int64_t n, const double lo[3], const double hi[3], int *dperm);

int launch_copy_probe(fvc_ctx *c, void *dst, const void *src, int64_t bytes);
/* a grid's FTLE values (i-major on the device) to host arrays in k, j, i order */
int copy_ftle_kji(fvc_ctx *c, const double *d_wt, const double *d_wot, const int32_t res[3], double *wt, double *wot);

int check_err(fvc_ctx *c, const char *what);

/* The choice between two builds of an integrator on an unstructured mesh by
 * the elements that a step crosses, crossings * dt.  The state machines keep
 * a lane's last element and cost nothing for a wave whose lanes cross
 * elements at different stages; every pass of theirs runs all phases' code,
 * so where most lanes cross elements anyway the straight-line walks, whose
 * waves walk together, are faster.  Both give the same bits.
 * FP64 RK4, machine over walks, 20 steps, at 0.1 / 0.2 / 0.3 / 0.45 / 1.2
 * elements a step: points ordered by element 1.26-1.44, 1.02-1.25, 0.89-1.11,
 * 0.69-0.93, 0.65-0.69; in random order 1.41-4.4, 1.1-3.2, 0.96-2.6,
 * 0.84-1.98, 0.71-1.37. */
inline bool rk4_walks(const fvc_ctx *c, double crossings, double dt) {
    return c->precision == 0 && c->mesh.mesh_type == 1 && !(crossings * fabs(dt) < 0.25);
}
/* AB2 and AB3, machine over walks, 300,000 points: 1.5-2.9 at 0.1, 1.07-1.58
 * at 0.45, 0.86-1.15 at 1.2; 75,000 in 3-D 1.05-1.4 at 0.45, in 2-D 1.04 at
 * 0.1 and 0.81 at 0.45; 3,000 points, one wave on a SIMD, 0.98-1.07 at 0.1
 * over 20 steps and 0.7-0.9 over 3, whose RK4 starts count. */
inline bool ab_machine(const fvc_ctx *c, double crossings, double dt, double span, int64_t count) {
    const bool full = count >= (c->mesh.dims == 3 ? 1 << 16 : 1 << 18);
    return full ? crossings * fabs(dt) < 0.45 : crossings * fabs(dt) < 0.1 && fabs(span) > 9.5 * fabs(dt);
}
/* after check_err: last_steps and last_idle of the launches since the last call */
inline void take_steps(fvc_ctx *c) {
    c->last_steps = (int64_t)(c->h_status->steps[0] - c->steps_seen[0]);
    c->last_idle = (int64_t)(c->h_status->steps[1] - c->steps_seen[1]);
    for (int k = 0; k < 2; k++) c->steps_seen[k] = c->h_status->steps[k];
}
/* order the main stream after the side stream's last launch / wait for it on the host */
int side_join(fvc_ctx *c);
int side_sync(fvc_ctx *c);
/* release an object's device memory and detach it from its context (the
 * handle stays valid for its *_destroy call only); no-ops when detached */
void particles_release(fvc_particles *p);
void ftle_release(fvc_ftle *f);
void batch_release(fvc_batch *b);
void server_release(fvc_server *s);
/* batches running over particle set p (released before p) */
void batches_release_on(fvc_ctx *c, fvc_particles *p);
void *scratch(fvc_ctx *c, size_t bytes);
/* bracket the hot kernel launch with events when timing is on */
inline void timing_begin(fvc_ctx *c) {
    if (c->timing) (void)hipEventRecord(c->ev0, c->stream);
}
inline void timing_end(fvc_ctx *c) {
    if (c->timing) (void)hipEventRecord(c->ev1, c->stream);
}
inline void timing_collect(fvc_ctx *c, int64_t steps) {
    if (!c->timing) return;
    float ms = 0.0f;
    if (hipEventSynchronize(c->ev1) == hipSuccess && hipEventElapsedTime(&ms, c->ev0, c->ev1) == hipSuccess) {
        c->t_ms += ms;
        c->t_launches++;
        c->t_steps += steps;
    }
}
} // namespace fvc

#define FVC_HIP(call)                                                                                                  \
    do {                                                                                                               \
        hipError_t e_ = (call);                                                                                        \
        if (e_ != hipSuccess) {                                                                                        \
            c->last_error = std::string(#call) + ": " + hipGetErrorString(e_);                                         \
            return e_ == hipErrorOutOfMemory ? FVC_E_NOMEM : FVC_E_HIP;                                                \
        }                                                                                                              \
    } while (0)
