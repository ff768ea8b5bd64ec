// batch.hip -- shared launches over several resident FP32-perturbation
// solvers of one scheme class, one RK step as a hipGraph.
//
// The reference has no serving mode; this is the device half of the
// continuous-batching service: the host side admits and retires solvers and
// re-forms the batch at step boundaries.
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "kernels_fp32p.hpp"
#include "lfm_hip.h"
#include "solver_state.hpp"

namespace lfm {

struct Batch {
    hipStream_t stream = nullptr;
    std::vector<Solver *> members;
    KArgs32 *d_args = nullptr;
    int2 *d_maps = nullptr;
    size_t maps_cap = 0, args_cap = 0;
    BatchMap map_cells{}, map_faces{};
    int nb_cells = 0, nb_faces = 0;
    int D = 2, solver = 0, minmod = 0, nstages = 0;
    bool visc = true;
    // inviscid M1 / M2 members with their second buffers and face slots: one
    // launch per stage, from one buffer into the other (side 1: the state is in
    // the second).  A graph ends in the first: one that holds an odd number of
    // stages takes its first as separate launches, which update in place (256 k
    // cells in four members: 15 us where a one-launch stage takes 8).
    bool fused = false;
    int side = 0;
    double A[5]{}, B[5]{};
    int separate = 0;      // first stages of each step that stay separate launches
    bool drop_dq = false;  // the step being enqueued is followed by another one of its graph
    int dq_mode(int rk) const { return (rk == 0 ? kDqZero : 0) | (drop_dq && rk == nstages - 1 ? kDqDrop : 0); }
    // one step, and kSteps of them for runs of many.  A graph launch costs
    // some 9 us beside its kernels, so the longer graph saves 8 us per step;
    // building it costs 0.6 (6 launches per step) to 1.3 ms (16), what it
    // saves in kManyAfter steps, and is done once that many were run (twice as
    // many after each time that it could not be had).
    static constexpr int kSteps = Solver::kGraphSteps;
    static_assert(kSteps % 2 == 0);
    static constexpr long kManyAfter = 128;
    hipGraph_t graph = nullptr, graph_many = nullptr;
    hipGraphExec_t exec = nullptr, exec_many = nullptr;
    long singles = 0;  // single-step launches since the members were set or a failure
    long many_after = kManyAfter;
    int64_t replayed_many = 0;  // steps taken by graphs of kSteps
    GraphBuild *building = nullptr;

    void drop_graphs() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (exec_many) (void)hipGraphExecDestroy(exec_many);
        if (graph_many) (void)hipGraphDestroy(graph_many);
        exec = exec_many = nullptr;
        graph = graph_many = nullptr;
        singles = 0;
        many_after = kManyAfter;
    }
    ~Batch() {
        drop_graphs();
        if (d_args) (void)hipFree(d_args);
        if (d_maps) (void)hipFree(d_maps);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

template <int D, int SOLVER, bool NT>
static void enqueue_fused(Batch *b, int rk, int flip) {
    const dim3 blk(256);
    if (rk == b->nstages - 1)
        launch(b, (stage_fused32_b<D, SOLVER, 1, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells, (float)b->A[rk],
               (float)b->B[rk], b->dq_mode(rk), flip);
    else
        launch(b, (stage_fused32_b<D, SOLVER, -1, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells,
               (float)b->A[rk], (float)b->B[rk], b->dq_mode(rk), flip);
}

template <int D, bool V, bool NT>
static void enqueue_step_nt(Batch *b) {
    const dim3 blk(256);
    for (int rk = 0; rk < b->nstages; rk++) {
        if (b->fused && rk >= b->separate) {
            b->solver == 0 ? enqueue_fused<D, 0, NT>(b, rk, b->side) : enqueue_fused<D, 1, NT>(b, rk, b->side);
            b->side ^= 1;
            continue;
        }
        // ghosts are refreshed by the update kernel (members join with fresh ghosts);
        // without viscosity solvers 0/1 consume no gradient or tensor
        if (V || b->solver == 2) {
            if (b->solver == 2 && b->minmod)
                launch(b, (grad_vis32_b<D, 2, V, true, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells);
            else if (b->solver == 2)
                launch(b, (grad_vis32_b<D, 0, V, true, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells);
            else
                launch(b, (grad_vis32_b<D, 0, V, false, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells);
        }
        switch (b->solver) {
        case 0: launch(b, (face_flux32_b<D, 0, V, NT>), dim3(b->nb_faces), blk, b->d_args, b->map_faces); break;
        case 1: launch(b, (face_flux32_b<D, 1, V, NT>), dim3(b->nb_faces), blk, b->d_args, b->map_faces); break;
        default: launch(b, (face_flux32_b<D, 2, V, NT>), dim3(b->nb_faces), blk, b->d_args, b->map_faces); break;
        }
        // the last stage's update also forms the step's compute_cfl partials
        if (rk == b->nstages - 1)
            launch(b, (cell_update32_b<D, 1, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells, (float)b->A[rk],
                   (float)b->B[rk], b->dq_mode(rk));
        else
            launch(b, (cell_update32_b<D, -1, NT>), dim3(b->nb_cells), blk, b->d_args, b->map_cells, (float)b->A[rk],
                   (float)b->B[rk], b->dq_mode(rk));
    }
    launch(b, cfl_final32_b, dim3((unsigned)b->members.size()), blk, b->d_args);
}

// one launch walks every member: NT by what they touch together
template <int D, bool V>
static void enqueue_step(Batch *b) {
    size_t bytes = 0;
    for (const Solver *s : b->members) bytes += s->stage_bytes;
    outgrows_cache(bytes) ? enqueue_step_nt<D, V, true>(b) : enqueue_step_nt<D, V, false>(b);
}

// n RK steps of the batch as a graph
static hipError_t build_steps(Batch *b, int n, hipGraph_t *graph, hipGraphExec_t *exec) {
    GraphBuild build;
    b->building = &build;
    b->side = 0;
    b->separate = n * b->nstages % 2;  // n is 1 or even
    for (int i = 0; i < n; i++) {
        b->drop_dq = i + 1 < n;
        if (b->D == 2)
            b->visc ? enqueue_step<2, true>(b) : enqueue_step<2, false>(b);
        else
            b->visc ? enqueue_step<3, true>(b) : enqueue_step<3, false>(b);
    }
    b->building = nullptr;
    return build.finish(graph, exec);
}

static int batch_set(Batch *b, lfm_solver *const *hs, int n) {
    // the one-launch stages' buffers of eligible members; a member without them
    // keeps the batch on separate launches
    for (int i = 0; i < n; i++)
        if (hs && hs[i] && hs[i]->impl && hs[i]->impl->fp32) (void)hs[i]->impl->ensure_alt32();
    if (b->exec) HIP_TRY(hipStreamSynchronize(b->stream));
    b->drop_graphs();
    b->members.clear();
    b->fused = false;
    if (n == 0) return LFM_OK;
    bool fused = true;
    std::vector<KArgs32> args;
    std::vector<int2> slot_c, slot_f;
    for (int i = 0; i < n; i++) {
        if (!hs[i] || !hs[i]->impl) return fail(LFM_EINVAL, "null solver in batch");
        Solver *s = hs[i]->impl.get();
        if (!s->fp32) return fail(LFM_EINVAL, "batched launches need FP32-perturbation solvers");
        if (!s->L.halo.empty()) return fail(LFM_EINVAL, "a partition with processor patches cannot join a batch");
        if (s->prm.have_res || s->prm.adjust_dt)
            return fail(LFM_EINVAL, "batched solvers run constant dt without residual output");
        if (i == 0) {
            b->D = s->L.D;
            b->solver = s->prm.solver;
            b->minmod = s->prm.minmod;
            b->nstages = s->nstages;
            b->visc = s->visc;
            for (int k = 0; k < 5; k++) {
                b->A[k] = s->A[k];
                b->B[k] = s->B[k];
            }
        } else if (s->L.D != b->D || s->prm.solver != b->solver || s->prm.minmod != b->minmod ||
                   s->nstages != b->nstages || s->visc != b->visc) {
            return fail(LFM_EINVAL, "batched solvers must share dimension, solver, minmod, rkOrder and whether "
                                    "they are viscous");
        }
        for (Solver *o : b->members)
            if (o == s) return fail(LFM_EINVAL, "solver listed twice in a batch");
        if (s->ghosts_stale) {
            s->bc();
            s->ghosts_stale = false;
        }
        if (int rc = s->ensure_keys(s->visc || s->prm.solver == 2)) return rc;
        HIP_TRY(hipStreamSynchronize(s->stream));
        b->members.push_back(s);
        args.push_back(*s->k32);
        args.back().q_alt = s->q_alt32;
        fused = fused && s->fused_ok && s->q_alt32 && !s->post_forces;
        auto add = [&](std::vector<int2> &slot, long count) {
            const int nb = (int)((count + 255) / 256);
            for (int k = 0; k < nb; k++) slot.push_back(make_int2(i, k));
        };
        add(slot_c, s->L.nc);
        add(slot_f, s->L.nf);
    }
    b->nb_cells = (int)slot_c.size();
    b->nb_faces = (int)slot_f.size();
    b->fused = fused && b->solver < 2 && !b->visc;
    const size_t nmap = slot_c.size() + slot_f.size();
    if (nmap > b->maps_cap) {
        if (b->d_maps) HIP_TRY(hipFree(b->d_maps));
        HIP_TRY(hipMalloc((void **)&b->d_maps, nmap * sizeof(int2)));
        b->maps_cap = nmap;
    }
    if ((size_t)n > b->args_cap) {
        if (b->d_args) HIP_TRY(hipFree(b->d_args));
        HIP_TRY(hipMalloc((void **)&b->d_args, n * sizeof(KArgs32)));
        b->args_cap = n;
    }
    b->map_cells.slot = b->d_maps;
    b->map_faces.slot = b->d_maps + slot_c.size();
    HIP_TRY(hipMemcpy(b->d_maps, slot_c.data(), slot_c.size() * sizeof(int2), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(b->d_maps + slot_c.size(), slot_f.data(), slot_f.size() * sizeof(int2), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(b->d_args, args.data(), n * sizeof(KArgs32), hipMemcpyHostToDevice));
    const hipError_t e = build_steps(b, 1, &b->graph, &b->exec);
    if (e != hipSuccess) {
        b->members.clear();
        return fail(LFM_EDEVICE, std::string("step graph: ") + hipGetErrorString(e));
    }
    return LFM_OK;
}

// the graph of kSteps steps, once the single ones have cost as much
static bool build_many(Batch *b) {
    if (b->singles < b->many_after) return false;
    if (build_steps(b, Batch::kSteps, &b->graph_many, &b->exec_many) == hipSuccess) return true;
    b->singles = 0;
    b->many_after *= 2;
    return false;
}

}  // namespace lfm

struct lfm_batch {
    lfm::Batch impl;
};

extern "C" {

int lfm_batch_create(lfm_batch **out) {
    if (!out) return lfm::fail(LFM_EINVAL, "null argument");
    auto *b = new lfm_batch;
    if (hipStreamCreateWithFlags(&b->impl.stream, hipStreamNonBlocking) != hipSuccess) {
        delete b;
        return lfm::fail(LFM_EDEVICE, "hipStreamCreateWithFlags failed");
    }
    *out = b;
    return LFM_OK;
}

int lfm_batch_destroy(lfm_batch *b) {
    if (!b) return LFM_OK;
    if (b->impl.stream) (void)hipStreamSynchronize(b->impl.stream);
    delete b;
    return LFM_OK;
}

int lfm_batch_set(lfm_batch *b, lfm_solver *const *solvers, int n) {
    if (!b || n < 0 || (n > 0 && !solvers)) return lfm::fail(LFM_EINVAL, "bad argument");
    return lfm::batch_set(&b->impl, solvers, n);
}

int lfm_batch_run(lfm_batch *b, int nsteps) {
    if (!b || nsteps < 0) return lfm::fail(LFM_EINVAL, "bad argument");
    if (b->impl.members.empty() || !b->impl.exec) return nsteps == 0 ? LFM_OK : lfm::fail(LFM_ESTATE, "empty batch");
    lfm::Batch &x = b->impl;
    for (int i = 0; i < nsteps;) {
        const bool many = nsteps - i >= x.kSteps && (x.exec_many || lfm::build_many(&x));
        const hipError_t e = hipGraphLaunch(many ? x.exec_many : x.exec, x.stream);
        if (e != hipSuccess) return lfm::fail(LFM_EDEVICE, std::string("hipGraphLaunch: ") + hipGetErrorString(e));
        i += many ? x.kSteps : 1;
        x.singles += many ? 0 : 1;
        x.replayed_many += many ? x.kSteps : 0;
    }
    for (lfm::Solver *s : b->impl.members) s->steps_done += nsteps;
    return LFM_OK;
}

int lfm_batch_replayed_steps(lfm_batch *b, int64_t *n) {
    if (!b || !n) return lfm::fail(LFM_EINVAL, "null argument");
    *n = b->impl.replayed_many;
    return LFM_OK;
}

int lfm_batch_synchronize(lfm_batch *b) {
    if (!b) return lfm::fail(LFM_EINVAL, "null handle");
    hipError_t e = hipStreamSynchronize(b->impl.stream);
    if (e != hipSuccess) return lfm::fail(LFM_EDEVICE, std::string("hipStreamSynchronize: ") + hipGetErrorString(e));
    return LFM_OK;
}

}  // extern "C"
