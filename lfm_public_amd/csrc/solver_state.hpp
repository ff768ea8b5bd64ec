// solver_state.hpp -- the device-resident state behind one lfm_solver handle.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <string>
#include <vector>

#include "graph_build.hpp"
#include "kernels_fp64.hpp"
#include "lfm_hip.h"
#include "mesh_builder.hpp"

namespace lfm {

// FP32-perturbation kernel arguments (defined in kernels_fp32p.hpp).
struct KArgs32;
// Post-processing state (averages, wall forces; defined in post.hip).
struct PostState;
void free_post(PostState *p);

int fail(int code, const std::string &msg);

// Returns the LFM_EDEVICE status (with the failing call and HIP's message
// recorded as the last error) from the enclosing function when a HIP call
// fails.
#define HIP_TRY(expr)                                                                            \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return fail(LFM_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));       \
    } while (0)

struct Solver {
    lfm_params prm{};
    SolverLayout L;
    Gas gas{};
    double A[5]{}, B[5]{};
    int nstages = 0;
    double dt = 0.0;
    bool fp32 = false;
    bool visc = true;  // mu != 0: the step forms the viscous terms

    int device = 0;  // the HIP device current when the handle was created
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double *h_scalar = nullptr;   // pinned host scratch (kScalars doubles, then kSmallRead bytes)
    static constexpr size_t kScalars = 64, kSmallRead = 128 << 10;
    // pinned ring for read-backs larger than kSmallRead, allocated by the
    // first one: two chunks and their events per worker
    struct ReadRing;
    ReadRing *read_ring = nullptr;
    const int32_t *d_comb = nullptr;  // L.comb on the device
    std::vector<void *> allocs;
    int64_t device_bytes = 0;
    // device memory of the set-up: small arrays share slabs, each filled on the
    // host and copied as a whole, so that creating a small solve does not take
    // an allocation and a copy per array
    int dev_alloc(void **p, size_t bytes);
    int dev_fill(void *p, const void *src, size_t bytes);  // src null: zeros
    int slab_flush();  // what was filled so far, before a kernel reads it
    // The gather entries (g_key, and g_oth where gradients are formed).  A solver
    // whose steps are one-launch stages reads neither: it gets them with the
    // first call that does (per-stage calls, FP32 compute_dt / compute_cfl,
    // separate launches of a batch or a group): 48 B per 3D cell, 32 per 2D cell.
    template <class Args>
    int build_gather_keys(Args &a, bool others, bool setup);
    bool keys_at_setup() const { return !fused_ok || prm.have_res; }
    int ensure_keys(bool others);
    int ensure_step_keys();
    char *slab = nullptr;
    size_t slab_used = 0, slab_copied = 0;
    std::unique_ptr<char[]> slab_host;

    // device scalars: [0] deltaT, [2..6] residual sums, [8] cfl, [9] dt min
    double *d_scalar = nullptr;
    double *d_res = nullptr, *d_cfl = nullptr, *d_dtmin = nullptr;
    double *d_dt_ptr() { return d_scalar; }

    KArgs k64{};
    KArgs32 *k32 = nullptr;       // owned via allocs-free host block

    // per-kernel-group timing with HIP events (lfm_profile_steps)
    // bc, grad_vis, face_flux, cell_update (and one-launch stages), cfl_dt
    // (final reductions), the last stage's update forming the CFL/dt extrema
    static constexpr int kProfGroups = 6;
    bool prof = false;
    std::vector<hipEvent_t> prof_ev;       // pairs (start, stop)
    std::vector<int> prof_grp;
    size_t prof_n = 0;
    void prof_mark(int grp, bool start);

    // halo lists on the device, one entry per L.halo neighbour
    struct HaloDev {
        int32_t *send_cells = nullptr;  // [n_send] local cells, ascending
        int32_t *recv_ghost = nullptr;  // [n_recv] ghost slot (combined index nc+g)
        int32_t *recv_src = nullptr;    // [n_recv] record in the received buffer
        int n_send = 0, n_recv = 0;
    };
    std::vector<HaloDev> halo_dev;
    bool halo_ready() const {
        for (const HaloNbr &h : L.halo)
            if (!h.imported) return false;
        return true;
    }
    int halo_index(int rank) const {
        for (size_t i = 0; i < L.halo.size(); i++)
            if (L.halo[i].rank == rank) return (int)i;
        return -1;
    }
    int halo_record(int kind) const {
        return ((kind & 1) ? L.D + 2 : 0) + ((kind & 2) ? 2 * L.D * L.D + 2 * L.D : 0);
    }
    int halo_pack(int ni, int kind, void *buf);
    int halo_unpack(int ni, int kind, const void *buf);
    int halo_upload_geometry();  // d, w of the faces after an import

    // post-processing (lfm_post_configure); post_forces mirrors
    // post->cfg.have_forces for the stage code
    PostState *post = nullptr;
    bool post_forces = false;
    // copies the boundary ghosts the wall forces read (their state as the
    // current stage's boundary fill left it)
    void post_snapshot();
    // the Mesh::solve post-processing after one step (time, averages, forces)
    int post_step();

    bool ghosts_stale = true;  // ghost states not derived from the current q
    double pending_A = 1.0;
    int pending_rk = 0;
    int64_t steps_done = 0;
    bool res_valid = false;

    ~Solver();

    // the end-of-step reduction: compute_dt (mode 0, min into out and, when
    // dt_dst is set, the deltaT the next step uses) or compute_cfl (mode 1)
    struct CflJob {
        int mode;
        double param;
        double *out, *dt_dst;
    };
    CflJob cfl_job(bool own_dt);
    bool cfl_fused = false;  // the last update of this step formed it

    // stage pieces on the handle's stream
    void bc();
    void gradvis(bool full, bool fin = false);
    void flux();
    // cfl: the update also forms that reduction from the updated cells (it
    // reads only a cell's own state and its faces' areas); not with res
    void update(double A, double B, int dq_mode, bool res, bool accumulate_res, const CflJob *cfl = nullptr);
    void cfl_dt(int mode, double param, double *out, double *dt_dst);
    // the final single-block reduction after an update that formed the
    // block extrema of a CFL job
    void cfl_final(const CflJob &job);
    void step();
    // pieces of step(): stage part A (ghost fill if stale, gradients and
    // viscous tensors), part B (fluxes, update), and the end-of-step CFL/dt
    // reduction (dt written to the own deltaT when own_dt).  stage_b of the
    // last stage forms that reduction in the update when fuse_cfl is set,
    // the stage computes no residual and the path is FP32 or 2D; end_step
    // then launches nothing.
    void stage_a(int rk);
    void stage_b(int rk, bool fuse_cfl = false, bool own_dt = true);
    // Inviscid M1 / M2 without halos or wall forces (fused_ok): stages from
    // fused_from() on are one launch each, reading one state buffer and
    // writing the other; after an odd count the two buffers swap roles, so
    // k32->q / k64.q always holds the state between steps.  The second buffer
    // is allocated by the first step that uses it (ensure_alt), so solvers
    // driven through the per-stage calls never hold it.
    bool fused_ok = false;
    float *q_alt32 = nullptr;
    double *q_alt64 = nullptr;
    bool ensure_alt() { return fp32 ? ensure_alt32() : ensure_alt64(); }
    bool have_alt() const { return fp32 ? q_alt32 != nullptr : q_alt64 != nullptr; }
    bool ensure_alt32();
    bool ensure_alt64();
    // the FP64 one-launch stage's slots (k64.pk or k64.sl_*, k64.s_perm), on
    // first use; the distinct face records found when the handle was created
    FaceTable<double> table64;
    FaceTable<float> table32;  // of the FP32 slots
    bool ensure_slots64();
    // bytes one stage touches; whether it outgrows the Infinity Cache, so that
    // its kernels stream what they touch once past the caches
    size_t stage_bytes = 0;
    bool stream_nt = false;
    bool records_nt = false;  // the FP64 gradient records alone do not stay in it
    void size_stage();
    bool sym64 = false;  // every record's weights allow flux_m1_sym
    // device memory for a set of arrays of one kind, all or none
    bool alloc_all(void **p, const size_t *bytes, int n);
    // per-cell face slots of the FP32 kernels (k32->pk or k32->sl_*), on
    // first use
    bool slots_failed = false;
    bool ensure_slots32();
    int fused_from() const;
    void stage_fused(int rk, bool from_alt);
    // the compute_cfl final reduction carried into the next step: when
    // defer_cfl is set (by a loop that steps again at once) and the next
    // step begins with a launch that can take it (carry_target), the last
    // stage leaves its per-block CFL maxima in the reduction scratch and
    // that launch reduces them in one extra block (no stage reads the CFL
    // at a fixed deltaT), which saves the single-block launch.  flush_cfl()
    // launches a carried reduction on its own; the loops call it when they
    // end.
    bool defer_cfl = false;
    bool cfl_pending = false;
    int carry_target() const;
    // the step is followed by another one in the same call
    bool drop_dq = false;
    int dq_mode(int rk) const { return (rk == 0 ? kDqZero : 0) | (drop_dq && rk == nstages - 1 ? kDqDrop : 0); }
    void final_or_carry(const CflJob &job);
    void flush_cfl();
    void end_step(bool own_dt);
    // n steps; with_post: the post-processing after each.  Long runs replay
    // kGraphSteps steps at a time as a graph.
    int run_steps(int n, bool with_post);
    static constexpr int kGraphSteps = 8;  // even: the state buffers' roles return
    struct StepGraph;
    StepGraph *step_graph = nullptr;
    GraphBuild *building = nullptr;  // set while launches become its nodes (launch)
    int graph_misses = 0;            // steps in a row whose launches were not the graph's
    long eager_launches = 0;         // since the last graph was built
    long graph_after = 0;            // and how many of them the next one waits for (0: kGraphAfter)
    int64_t replayed_steps = 0;
    bool graph_ready();
    bool graph_build();
    void free_step_graph();
    void zero_state_for_step();

    int get_field(int which, double *out);
    // the state in original cell order, components one after the other
    int read_state(double *out);
    // one per-cell array, times f (root: its square root), in that order
    int read_cells(const double *dev, double f, bool root, double *out);
    template <typename T, class Fill, class Sink>
    int stream_out(size_t n, const Fill &fill, const Sink &sink);
    void free_read_ring();
    int set_field(int which, const double *in);
    int check_finite(int64_t *n_bad);
    // the same count with its per-block partials in the library's static
    // device scratch instead of an allocated counter
    int check_finite_noalloc(int64_t *n_bad);
};

int create_fp32p(Solver *s);
void free_k32(KArgs32 *k);
int get_field32(Solver *s, int which, double *out);
int nonfinite32(Solver *s, unsigned long long *d);
// FP64 conservation integrals sum_c V_c q_c into out_dev[0..D+1] (device)
int integrals(Solver *s, double *out_dev);
int integrals64(Solver *s, double *out_dev);

}  // namespace lfm

// opaque handle of the C ABI
struct lfm_solver {
    std::unique_ptr<lfm::Solver> impl;
};
