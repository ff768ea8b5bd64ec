// solver.hip -- device state, launches and the C ABI (include/lfm_hip.h).
//
// One lfm_solver holds one partition (both reference submeshes) resident in
// HBM in SoA layout and drives the stage kernels on its own HIP stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "kernels_fp64.hpp"
#include "kernels_fp32p.hpp"
#include "lfm_hip.h"
#include "mesh_builder.hpp"
#include "solver_state.hpp"

namespace lfm {

thread_local std::string g_last_error;

int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}

// records of the FP64 geometry table: both orientations of them are at most
// 192 KiB, which stay in an XCD's 4 MiB L2 beside the gathered states
static constexpr int kMaxTable64 = 2048;
static constexpr int kBlock = 256;
static inline int nblocks(long n) { return (int)((n + kBlock - 1) / kBlock); }

static constexpr size_t kSlab = 1 << 20;
int Solver::dev_alloc(void **p, size_t bytes) {
    constexpr size_t kShare = 128 << 10, kAlign = 256;
    const size_t need = (bytes + kAlign - 1) / kAlign * kAlign;
    if (need > kShare) {
        HIP_TRY(hipMalloc(p, bytes));
        allocs.push_back(*p);
    } else {
        if (!slab || slab_used + need > kSlab) {
            if (int rc = slab_flush()) return rc;
            slab = nullptr;
            HIP_TRY(hipMalloc((void **)&slab, kSlab));
            allocs.push_back(slab);
            slab_used = slab_copied = 0;
            slab_host.reset(new char[kSlab]);
        }
        *p = slab + slab_used;
        slab_used += need;
    }
    device_bytes += (int64_t)bytes;
    return 0;
}

int Solver::dev_fill(void *p, const void *src, size_t bytes) {
    const size_t at = (size_t)((char *)p - slab);
    if (slab && (char *)p >= slab && at >= slab_copied && at + bytes <= slab_used)
        src ? std::memcpy(slab_host.get() + at, src, bytes) : std::memset(slab_host.get() + at, 0, bytes);
    else if (src)
        HIP_TRY(hipMemcpy(p, src, bytes, hipMemcpyHostToDevice));
    else
        HIP_TRY(hipMemset(p, 0, bytes));
    return 0;
}

int Solver::slab_flush() {
    if (slab && slab_used > slab_copied)
        HIP_TRY(hipMemcpy(slab + slab_copied, slab_host.get() + slab_copied, slab_used - slab_copied,
                          hipMemcpyHostToDevice));
    slab_copied = slab_used;
    return 0;
}

template <typename T>
static int dev_upload(Solver *s, T **dst, const T *src, size_t n) {
    if (n == 0) {
        *dst = nullptr;
        return 0;
    }
    if (int rc = s->dev_alloc((void **)dst, n * sizeof(T))) return rc;
    return src ? s->dev_fill(*dst, src, n * sizeof(T)) : 0;
}

template <typename T>
static int dev_zeros(Solver *s, T **dst, size_t n) {
    if (n == 0) {
        *dst = nullptr;
        return 0;
    }
    if (int rc = s->dev_alloc((void **)dst, n * sizeof(T))) return rc;
    return s->dev_fill(*dst, nullptr, n * sizeof(T));
}

// The fixed-width gather entries of an argument block whose lists are on the
// device.  At set-up among its arrays (on the null stream, as the uploads);
// later on the handle's stream, which is waited for (a batch or a group reads
// them on its own).
template <class Args>
int Solver::build_gather_keys(Args &a, bool others, bool setup) {
    const size_t n = keys_len(L.D, L.nc) * sizeof(int32_t);
    void *key = (void *)a.g_key, *oth = (void *)a.g_oth;
    for (void **p : {&key, &oth}) {
        if (*p || (p == &oth && !others)) continue;
        if (setup) {
            if (int rc = dev_alloc(p, n)) return rc;
        } else if (!alloc_all(p, &n, 1)) {
            return fail(LFM_EDEVICE, "no device memory for the gather entries");
        }
    }
    if (setup)
        if (int rc = slab_flush()) return rc;
    auto build = L.D == 2 ? build_keys<2> : build_keys<3>;
    hipLaunchKernelGGL(build, dim3(nblocks(L.nc)), dim3(kBlock), 0, setup ? nullptr : stream, L.nc, a.g_off, a.g_ent,
                       a.fP, a.fN, (int32_t *)key, (int32_t *)oth);
    HIP_TRY(hipGetLastError());
    if (!setup) HIP_TRY(hipStreamSynchronize(stream));
    a.g_key = (const int32_t *)key;
    a.g_oth = (const int32_t *)oth;
    return 0;
}
template int Solver::build_gather_keys<KArgs32>(KArgs32 &, bool, bool);

int Solver::ensure_keys(bool others) {
    const int32_t *key = fp32 ? k32->g_key : k64.g_key, *oth = fp32 ? k32->g_oth : k64.g_oth;
    if (key && (oth || !others)) return LFM_OK;
    return fp32 ? build_gather_keys(*k32, others, false) : build_gather_keys(k64, others, false);
}

int Solver::ensure_step_keys() {
    if (nstages > 0 && fused_ok && ensure_alt() && fused_from() == 0) return LFM_OK;
    return ensure_keys(visc || prm.solver == 2);
}

Solver::~Solver() {
    free_step_graph();
    for (void *p : allocs) (void)hipFree(p);
    if (k32) free_k32(k32);
    free_post(post);
    free_read_ring();
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
    if (h_scalar) (void)hipHostFree(h_scalar);
}

// ---------------------------------------------------------------------------
// creation
// ---------------------------------------------------------------------------
static int create_fp64(Solver *s) {
    const SolverLayout &L = s->L;
    const int D = L.D;
    const size_t nc = L.nc, ntot = (size_t)L.nc + L.ng, nf = L.nf;
    KArgs &a = s->k64;
    std::memset(&a, 0, sizeof(a));
    a.nc = L.nc;
    a.nsm0 = L.nsm0;
    a.ng = L.ng;
    a.nf = L.nf;
    a.ng_bnd = L.ng_bnd;
    a.ntot = (int)ntot;
    int rc = 0;
    rc |= dev_upload(s, (int32_t **)&a.fP, L.fP.data(), nf);
    rc |= dev_upload(s, (int32_t **)&a.fN, L.fN.data(), nf);
    {
        // S as one record per face ([nf][D])
        std::vector<double> Sr((size_t)D * nf);
        for (size_t f = 0; f < nf; f++)
            for (int k = 0; k < D; k++) Sr[f * D + k] = L.S[(size_t)k * nf + f];
        rc |= dev_upload(s, (double **)&a.S, Sr.data(), Sr.size());
    }
    rc |= dev_upload(s, (double **)&a.d, L.d.data(), (size_t)D * nf);
    rc |= dev_upload(s, (double **)&a.w, L.w.data(), nf);
    rc |= dev_upload(s, (int32_t **)&a.g_off, L.g_off.data(), nc + 1);
    rc |= dev_upload(s, (int32_t **)&a.g_ent, L.g_ent.data(), L.g_ent.size());
    rc |= dev_upload(s, (int32_t **)&a.s_off, L.s_off.data(), nc + 1);
    rc |= dev_upload(s, (int32_t **)&a.s_ent, L.s_ent.data(), L.s_ent.size());
    rc |= dev_upload(s, (int32_t **)&a.ghost_cell, L.ghost_cell.data(), L.ng);
    rc |= dev_upload(s, (int32_t **)&a.ghost_role, L.ghost_role.data(), L.ng);
    rc |= dev_upload(s, (double **)&a.vinv, L.vinv.data(), nc);
    if (std::any_of(L.sigma.begin(), L.sigma.end(), [](double v) { return v != 0.0; }))
        rc |= dev_upload(s, (double **)&a.sigma, L.sigma.data(), nc);
    if (!L.smag.empty()) rc |= dev_upload(s, (double **)&a.smag, L.smag.data(), nc);
    rc |= dev_zeros(s, &a.q, (size_t)(D + 2) * ntot);
    rc |= dev_zeros(s, &a.dq, (size_t)(D + 2) * nc);
    rc |= dev_zeros(s, &a.res_cell, (size_t)(D + 2) * nc);
    // gradient records (GradRec64): dudx, dTdx and (M2AUSM) the rho, p and U
    // gradients; solver 2 without minmodExists reads their never-computed
    // (zero) slots
    const bool rg = s->prm.solver == 2;
    a.gstride = grad_record_stride64(D, rg);
    rc |= dev_zeros(s, &a.dudx, (size_t)a.gstride * ntot);
    // tauMC / sigmaU are kept only for the halo payload of a partition; the
    // face kernel otherwise recomputes them from dudx
    if (!L.halo.empty()) {
        rc |= dev_zeros(s, &a.tauMC, (size_t)D * D * ntot);
        rc |= dev_zeros(s, &a.sigmaU, (size_t)D * ntot);
    }
    if (rc) return LFM_EDEVICE;
    a.dTdx = a.dudx + D * D;
    if (rg) {
        a.rho_grad = a.dudx + D * D + D;
        a.p_grad = a.dudx + D * D + 2 * D;
        a.U_grad = a.dudx + D * D + 3 * D;
    }
    rc |= dev_zeros(s, &a.frhs, (size_t)(D + 2) * nf);
    const size_t npart = (size_t)nblocks((long)std::max(nc, nf)) * (D + 2) + 16;
    rc |= dev_zeros(s, &a.partial, npart);
    rc |= dev_zeros(s, &s->d_scalar, 16);
    if (rc) return LFM_EDEVICE;
    a.dt = s->d_scalar + 0;
    s->d_res = s->d_scalar + 2;  // D+2 <= 5 slots: [2, 7)
    s->d_cfl = s->d_scalar + 8;
    s->d_dtmin = s->d_scalar + 9;
    const Gas &g = s->gas;
    a.gamma = g.gamma;
    a.gm1 = g.gm1;
    a.R_inv = g.R_inv;
    a.mu = g.mu;
    a.cp = g.cp;
    a.pr_inv = g.pr_inv;
    a.p_inf = g.p_inf;
    a.T_inf = g.T_inf;
    a.rho_inf = g.rho_inf;
    a.E_inf = g.E_inf;
    for (int k = 0; k < 3; k++) a.U_inf[k] = g.U_inf[k];
    // initial state into q (cells part, as cell records) and deltaT
    {
        std::vector<double> q0((size_t)(D + 2) * ntot, 0.0);
        for (int k = 0; k < D + 2; k++)
            for (size_t c = 0; c < nc; c++) q0[q64_index(k, c, ntot)] = L.q0[(size_t)k * nc + c];
        if (int rc = s->dev_fill(a.q, q0.data(), q0.size() * sizeof(double))) return rc;
    }
    if (int rc = s->dev_fill(s->d_scalar, &s->dt, sizeof(double))) return rc;
    // one-launch stages; a cell that is its own neighbour (a cyclic pair one
    // cell apart) has more gather entries than slots and keeps the launches
    // that walk the list
    s->fused_ok = !s->visc && s->prm.solver < 2 && L.halo.empty() && !own_neighbour(L);
    a.more_faces = max_entries(L) > (D == 2 ? GatherUnroll<2>::value : GatherUnroll<3>::value);
    if (s->keys_at_setup() && s->build_gather_keys(a, s->visc || s->prm.solver == 2, true)) return LFM_EDEVICE;
    if (s->fused_ok) {
        // records in both orientations and a placeholder's fit above the
        // cell index; kMaxTable64 keeps the table in an XCD's L2
        a.pk_shift = index_bits((long)ntot);
        const long fit = ((1L << (32 - a.pk_shift)) - 1) / 2;
        s->table64 = face_table<double>(L, (int)std::min<long>(fit, kMaxTable64));
    }
    return 0;
}

// ---------------------------------------------------------------------------
// FP64 launches
// ---------------------------------------------------------------------------
template <int D>
static void launch_bc64(Solver *s) {
    if (s->L.ng) launch(s, bc_fill<D>, dim3(nblocks(s->L.ng)), dim3(kBlock), s->k64);
}

template <int D, bool V, bool NT, bool RNT>
static void launch_gradvis64_nt(Solver *s) {
    const int nb = nblocks(s->L.nc);
    if (s->prm.solver == 2 && s->prm.minmod)
        launch(s, (grad_vis<D, 2, V, true, NT, RNT>), dim3(nb), dim3(kBlock), s->k64);
    else if (s->prm.solver == 2)
        launch(s, (grad_vis<D, 0, V, true, NT, RNT>), dim3(nb), dim3(kBlock), s->k64);
    else
        launch(s, (grad_vis<D, 0, V, false, NT, RNT>), dim3(nb), dim3(kBlock), s->k64);
}

template <int D, bool V>
static void launch_gradvis64_v(Solver *s) {
    if constexpr (V)  // without viscosity the records are not written whole
        if (s->records_nt) return launch_gradvis64_nt<D, V, true, true>(s);
    s->stream_nt ? launch_gradvis64_nt<D, V, true, false>(s) : launch_gradvis64_nt<D, V, false, false>(s);
}

// full: every tensor calc_VIS forms (the per-stage entry point); otherwise
// only what the step consumes (nothing for solvers 0/1 when mu = 0)
template <int D>
static void launch_gradvis64(Solver *s, bool full) {
    if (full || s->visc)
        launch_gradvis64_v<D, true>(s);
    else if (s->prm.solver == 2)
        launch_gradvis64_v<D, false>(s);
}

template <int D, bool V, bool ST, bool NT>
static void launch_flux64_nt(Solver *s) {
    const int nb = nblocks(s->L.nf);
    switch (s->prm.solver) {
    case 0: launch(s, (face_flux<D, 0, V, ST, NT>), dim3(nb), dim3(kBlock), s->k64); break;
    case 1: launch(s, (face_flux<D, 1, V, ST, NT>), dim3(nb), dim3(kBlock), s->k64); break;
    default: launch(s, (face_flux<D, 2, V, ST, NT>), dim3(nb), dim3(kBlock), s->k64); break;
    }
}

template <int D, bool V, bool ST>
static void launch_flux64_v(Solver *s) {
    s->stream_nt ? launch_flux64_nt<D, V, ST, true>(s) : launch_flux64_nt<D, V, ST, false>(s);
}

template <int D>
static void launch_flux64(Solver *s) {
    if (s->visc)
        s->k64.tauMC ? launch_flux64_v<D, true, true>(s) : launch_flux64_v<D, true, false>(s);
    else
        launch_flux64_v<D, false, false>(s);
}

template <int D, bool NT>
static void launch_update64_nt(Solver *s, double A, double B, int dq_mode, bool res, bool accumulate_res,
                               const Solver::CflJob *cfl) {
    const int nb = nblocks(s->L.nc);
    if (res) {
        launch(s, (cell_update<D, true, -1, NT>), dim3(nb), dim3(kBlock), s->k64, A, B, dq_mode, 0.0);
        launch(s, reduce_sum, dim3(1), dim3(kBlock), s->k64.partial, nb, D + 2, s->d_res, (int)accumulate_res);
    } else if (cfl && cfl->mode == 0) {
        launch(s, (cell_update<D, false, 0, NT>), dim3(nb), dim3(kBlock), s->k64, A, B, dq_mode, cfl->param);
    } else if (cfl) {
        launch(s, (cell_update<D, false, 1, NT>), dim3(nb), dim3(kBlock), s->k64, A, B, dq_mode, cfl->param);
    } else {
        launch(s, (cell_update<D, false, -1, NT>), dim3(nb), dim3(kBlock), s->k64, A, B, dq_mode, 0.0);
    }
}

template <int D>
static void launch_update64(Solver *s, double A, double B, int dq_mode, bool res, bool accumulate_res,
                            const Solver::CflJob *cfl) {
    s->stream_nt ? launch_update64_nt<D, true>(s, A, B, dq_mode, res, accumulate_res, cfl)
                 : launch_update64_nt<D, false>(s, A, B, dq_mode, res, accumulate_res, cfl);
}

template <int D>
static void launch_cfl_dt64(Solver *s, int mode, double param, double *out, double *dt_dst) {
    const int nb = nblocks(s->L.nc);
    if (mode == 0) {
        launch(s, (cfl_dt_cells<D, 0>), dim3(nb), dim3(kBlock), s->k64, param);
        launch(s, cfl_dt_final<0>, dim3(1), dim3(kFinalBlock), s->k64.partial, nb, out, dt_dst);
    } else {
        launch(s, (cfl_dt_cells<D, 1>), dim3(nb), dim3(kBlock), s->k64, param);
        launch(s, cfl_dt_final<1>, dim3(1), dim3(kFinalBlock), s->k64.partial, nb, out, dt_dst);
    }
}

int integrals64(Solver *s, double *out_dev) {
    const int nb = nblocks(s->L.nc);
    if (s->L.D == 2)
        launch(s, integrals64<2>, dim3(nb), dim3(kBlock), s->k64);
    else
        launch(s, integrals64<3>, dim3(nb), dim3(kBlock), s->k64);
    launch(s, reduce_sum, dim3(1), dim3(kBlock), s->k64.partial, nb, s->L.D + 2, out_dev, 0);
    return 0;
}

template <int D, int SOLVER, bool PK, bool SYM, bool NT>
static void launch_fused64_nt(Solver *s, double A, double B, int dq_mode, const KArgs &a, double *qout,
                             const Solver::CflJob *cfl, bool fin) {
    const int nb = nblocks(s->L.nc);
    if (!cfl)
        launch(s, (stage_fused64<D, SOLVER, -1, PK, SYM, NT>), dim3(nb + (fin ? 1 : 0)), dim3(kBlock), a, qout, A, B,
               dq_mode, 0.0, fin ? nb : 0, s->d_cfl);
    else if (cfl->mode == 0)
        launch(s, (stage_fused64<D, SOLVER, 0, PK, SYM, NT>), dim3(nb), dim3(kBlock), a, qout, A, B, dq_mode,
               cfl->param, 0, s->d_cfl);
    else
        launch(s, (stage_fused64<D, SOLVER, 1, PK, SYM, NT>), dim3(nb), dim3(kBlock), a, qout, A, B, dq_mode,
               cfl->param, 0, s->d_cfl);
}

template <int D, int SOLVER, bool PK, bool SYM>
static void launch_fused64_v(Solver *s, double A, double B, int dq_mode, const KArgs &a, double *qout,
                             const Solver::CflJob *cfl, bool fin) {
    s->stream_nt ? launch_fused64_nt<D, SOLVER, PK, SYM, true>(s, A, B, dq_mode, a, qout, cfl, fin)
                 : launch_fused64_nt<D, SOLVER, PK, SYM, false>(s, A, B, dq_mode, a, qout, cfl, fin);
}

// fin: the launch also reduces the previous step's CFL maxima (left in
// a.partial) into d_cfl, in one extra block
template <int D>
static void launch_stage_fused64(Solver *s, double A, double B, int dq_mode, const double *qin, double *qout,
                                 const Solver::CflJob *cfl, bool fin) {
    KArgs a = s->k64;
    a.q = const_cast<double *>(qin);
    if (s->prm.solver == 1)
        a.pk ? launch_fused64_v<D, 1, true, false>(s, A, B, dq_mode, a, qout, cfl, fin)
             : launch_fused64_v<D, 1, false, false>(s, A, B, dq_mode, a, qout, cfl, fin);
    else if (a.pk)
        s->sym64 ? launch_fused64_v<D, 0, true, true>(s, A, B, dq_mode, a, qout, cfl, fin)
                 : launch_fused64_v<D, 0, true, false>(s, A, B, dq_mode, a, qout, cfl, fin);
    else
        launch_fused64_v<D, 0, false, false>(s, A, B, dq_mode, a, qout, cfl, fin);
}

// dispatch helpers over dimension
#define LFM_DISPATCH_D(s, call2, call3) \
    do {                                \
        if ((s)->L.D == 2) {            \
            call2;                      \
        } else {                        \
            call3;                      \
        }                               \
    } while (0)

// ---------------------------------------------------------------------------
// precision-generic stage pieces
// ---------------------------------------------------------------------------
void Solver::bc() {
    if (fp32) {
        LFM_DISPATCH_D(this, launch_bc32<2>(this), launch_bc32<3>(this));
    } else {
        LFM_DISPATCH_D(this, launch_bc64<2>(this), launch_bc64<3>(this));
    }
}

void Solver::gradvis(bool full, bool fin) {
    if (fp32) {
        LFM_DISPATCH_D(this, launch_gradvis32<2>(this, full, fin), launch_gradvis32<3>(this, full, fin));
    } else {
        LFM_DISPATCH_D(this, launch_gradvis64<2>(this, full), launch_gradvis64<3>(this, full));
    }
}

void Solver::flux() {
    if (fp32) {
        LFM_DISPATCH_D(this, launch_flux32<2>(this), launch_flux32<3>(this));
    } else {
        LFM_DISPATCH_D(this, launch_flux64<2>(this), launch_flux64<3>(this));
    }
}

void Solver::update(double A, double B, int dq_mode, bool res, bool accumulate_res, const CflJob *cfl) {
    if (fp32) {
        LFM_DISPATCH_D(this, launch_update32<2>(this, A, B, dq_mode, res, accumulate_res, cfl),
                       launch_update32<3>(this, A, B, dq_mode, res, accumulate_res, cfl));
    } else {
        LFM_DISPATCH_D(this, launch_update64<2>(this, A, B, dq_mode, res, accumulate_res, cfl),
                       launch_update64<3>(this, A, B, dq_mode, res, accumulate_res, cfl));
    }
}

// the single-block final reduction of the block extrema an update with a
// CFL job left in the reduction scratch (shared by both precision paths)
void Solver::cfl_final(const CflJob &job) {
    const int nb = nblocks(L.nc);
    if (job.mode == 0)
        launch(this, cfl_dt_final<0>, dim3(1), dim3(kFinalBlock), k64.partial, nb, job.out, job.dt_dst);
    else
        launch(this, cfl_dt_final<1>, dim3(1), dim3(kFinalBlock), k64.partial, nb, job.out, job.dt_dst);
}

void Solver::cfl_dt(int mode, double param, double *out, double *dt_dst) {
    if (fp32) {
        LFM_DISPATCH_D(this, launch_cfl_dt32<2>(this, mode, param, out, dt_dst),
                       launch_cfl_dt32<3>(this, mode, param, out, dt_dst));
    } else {
        LFM_DISPATCH_D(this, launch_cfl_dt64<2>(this, mode, param, out, dt_dst),
                       launch_cfl_dt64<3>(this, mode, param, out, dt_dst));
    }
}

void Solver::prof_mark(int grp, bool start) {
    if (!prof) return;
    if (prof_n >= prof_ev.size()) return;
    (void)hipEventRecord(prof_ev[prof_n], stream);
    prof_grp[prof_n] = start ? grp : -1 - grp;
    prof_n++;
}

void Solver::stage_a(int rk) {
    (void)rk;
    // the update kernel refreshes the boundary ghosts; a full fill is needed
    // only after the state was set from outside
    if (ghosts_stale) {
        prof_mark(0, true);
        bc();
        prof_mark(0, false);
        ghosts_stale = false;
    }
    // a carried CFL reduction is taken by the step's first gradient launch
    const bool fin = cfl_pending && carry_target() == 2;
    if (fin) cfl_pending = false;
    prof_mark(1, true);
    gradvis(false, fin);
    prof_mark(1, false);
}

Solver::CflJob Solver::cfl_job(bool own_dt) {
    if (prm.adjust_dt) return CflJob{0, prm.max_co, d_dtmin, own_dt ? d_dt_ptr() : nullptr};
    return CflJob{1, dt, d_cfl, nullptr};
}

void Solver::stage_b(int rk, bool fuse_cfl, bool own_dt) {
    const bool res = prm.have_res != 0 && rk == 0;
    prof_mark(2, true);
    flux();
    prof_mark(2, false);
    // the update refreshes the boundary ghosts from the updated cells; the
    // wall forces after this step read them as this stage began
    if (post_forces && rk == nstages - 1) post_snapshot();
    // fused where measured faster: the FP64 3D update runs at 4 waves per
    // SIMD, where the appended slot gathers cost more than their own launch
    // (4.2 M-cell O-grid: 1.760 -> 1.779 ms per step; 2D and FP32 gain
    // 7-11 us per step on 1 M cells)
    if (fuse_cfl && rk == nstages - 1 && !res && (fp32 || L.D == 2)) {
        const CflJob job = cfl_job(own_dt);
        prof_mark(5, true);
        update(A[rk], B[rk], dq_mode(rk), false, false, &job);
        prof_mark(5, false);
        final_or_carry(job);
        cfl_fused = true;
    } else {
        prof_mark(3, true);
        update(A[rk], B[rk], dq_mode(rk), res, false);
        prof_mark(3, false);
    }
}

void Solver::end_step(bool own_dt) {
    if (cfl_fused) {
        cfl_fused = false;
    } else {
        prof_mark(4, true);
        const CflJob job = cfl_job(own_dt);
        cfl_dt(job.mode, job.param, job.out, job.dt_dst);
        prof_mark(4, false);
    }
    steps_done++;
    if (prm.have_res) res_valid = true;
}

// a face table's record numbers on the device (freed by the caller), nullptr
// where memory cannot be had
static void *upload_records(const std::vector<uint16_t> &rec) {
    void *p = nullptr;
    if (hipMalloc(&p, rec.size() * sizeof(uint16_t)) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (hipMemcpy(p, rec.data(), rec.size() * sizeof(uint16_t), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(p);
        return nullptr;
    }
    return p;
}

// the per-cell face slots (each cell's first GatherUnroll gather entries:
// other cell, area vector, weight), read by the one-launch stages and the 3D
// FP32 gradient kernel; allocated on first use and filled from the gather list
// on the handle's stream.  When memory cannot be had the gradients read the
// gather entries and the face arrays and the step runs the separate launches,
// which gives the same bits.
bool Solver::ensure_slots32() {
    if (!fp32 || slots_failed) return false;
    if (k32->pk || k32->sl_nb) return true;
    const int D = L.D, U = D == 2 ? GatherUnroll<2>::value : GatherUnroll<3>::value, nt = table32.n;
    void *p[3] = {nullptr, nullptr, nullptr}, *rec = nullptr;
    slots_failed = true;
    if (nt) {
        // each record with S as P sees it, then as N does, and a placeholder's
        std::vector<float> tab((size_t)(2 * nt + 1) * 4, 0.f);
        bool half = true;
        for (int i = 0; i < 2 * nt; i++) {
            const float w = table32.w[i / 2];
            for (int k = 0; k < D; k++) {
                const float x = table32.S[(size_t)(i / 2) * D + k];
                tab[(size_t)i * 4 + k] = i % 2 ? -x : x;
            }
            tab[(size_t)i * 4 + D] = w;
            half = half && w == 0.5f;
        }
        tab[(size_t)2 * nt * 4 + D] = 0.5f;
        const size_t bytes[2] = {pk_len(D, L.nc, U) * sizeof(uint32_t), tab.size() * sizeof(float)};
        if (!alloc_all(p, bytes, 2)) return false;
        rec = upload_records(table32.rec);
        if (!rec || hipMemcpy(p[1], tab.data(), bytes[1], hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipGetLastError();
            if (rec) (void)hipFree(rec);
            return false;
        }
        k32->pk_half = half;
    } else {
        const size_t bytes[3] = {slot_array_len(L.nc, U, 1) * sizeof(int32_t),
                                 slot_array_len(L.nc, U, D) * sizeof(float),
                                 slot_array_len(L.nc, U, 1) * sizeof(float)};
        if (!alloc_all(p, bytes, 3)) return false;
    }
    uint32_t *pk = nt ? (uint32_t *)p[0] : nullptr;
    int32_t *nb = nt ? nullptr : (int32_t *)p[0];
    float *sS = nt ? nullptr : (float *)p[1], *sw = nt ? nullptr : (float *)p[2];
    LFM_DISPATCH_D(this, launch_build_slots32<2>(this, (const uint16_t *)rec, 2 * nt, pk, nb, sS, sw),
                   launch_build_slots32<3>(this, (const uint16_t *)rec, 2 * nt, pk, nb, sS, sw));
    if (rec) {
        (void)hipStreamSynchronize(stream);
        (void)hipFree(rec);
    }
    table32 = FaceTable<float>();
    k32->pk = pk;
    k32->pk_tab = nt ? (const float *)p[1] : nullptr;
    k32->sl_nb = nb;
    k32->sl_S = sS;
    k32->sl_w = sw;
    slots_failed = false;
    return true;
}

// What one RK stage touches, and whether its kernels mark what they touch once
// as non-temporal.
void Solver::size_stage() {
    StageShape sh;
    sh.D = L.D;
    sh.word = fp32 ? sizeof(float) : sizeof(double);
    sh.nc = L.nc;
    sh.nf = L.nf;
    sh.one_launch = fused_ok;
    sh.packed = fp32 ? table32.n > 0 : table64.n > 0;
    if (visc || prm.solver == 2) sh.grad_values = fp32 ? k32->gstride : k64.gstride;
    stage_bytes = stage_footprint(sh);
    stream_nt = outgrows_cache(stage_bytes);
    records_nt = stream_nt && sh.nc * sh.grad_values * sh.word > (size_t)190 * 1000 * 1000;
}

bool Solver::alloc_all(void **p, const size_t *bytes, int n) {
    for (int i = 0; i < n; i++)
        if (hipMalloc(&p[i], bytes[i]) != hipSuccess) {
            (void)hipGetLastError();
            for (int k = 0; k < i; k++) (void)hipFree(p[k]);
            return false;
        }
    for (int i = 0; i < n; i++) {
        allocs.push_back(p[i]);
        device_bytes += (int64_t)bytes[i];
    }
    return true;
}

// the FP64 one-launch stage's slots: packed words over the geometry table
// where the mesh has few distinct face records, else each slot's key, area
// vector and weight
bool Solver::ensure_slots64() {
    if (k64.s_perm) return true;
    const int D = L.D, U = D == 2 ? GatherUnroll<2>::value : GatherUnroll<3>::value;
    const size_t words = slot_array_len(L.nc, U, 1) * sizeof(int32_t), perm = (size_t)L.nc * sizeof(int32_t);
    void *p[4] = {nullptr, nullptr, nullptr, nullptr}, *rec = nullptr;
    const int nt = table64.n;
    std::vector<double> tab;
    if (nt) {
        // each record as P sees it, then as N does (flux_m1), and a
        // placeholder's; |S| summed and rooted as the kernels would
        tab.assign((size_t)(2 * nt + 1) * kTabRec64, 0.0);
        sym64 = true;
        for (int i = 0; i < 2 * nt; i++) {
            double *r = &tab[(size_t)i * kTabRec64], m = 0.0;
            const double w = table64.w[i / 2], omw = 1.0 - w;
            for (int k = 0; k < D; k++) {
                const double x = table64.S[(size_t)(i / 2) * D + k];
                m += x * x;
                r[k] = i % 2 ? -x : x;
            }
            r[D] = std::sqrt(m);
            r[D + 1] = i % 2 ? omw : w;
            r[D + 2] = i % 2 ? w : omw;
            sym64 = sym64 && 1.0 - omw == w;
        }
        double *r = &tab[(size_t)2 * nt * kTabRec64];
        r[0] = r[D] = 1.0;
        r[D + 1] = r[D + 2] = 0.5;
        const size_t bytes[3] = {words, tab.size() * sizeof(double), perm};
        if (!alloc_all(p, bytes, 3)) return false;
        rec = upload_records(table64.rec);
        if (!rec || hipMemcpy(p[1], tab.data(), bytes[1], hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipGetLastError();
            if (rec) (void)hipFree(rec);
            return false;
        }
    } else {
        const size_t bytes[4] = {words, slot_array_len(L.nc, U, D) * sizeof(double),
                                 slot_array_len(L.nc, U, 1) * sizeof(double), perm};
        if (!alloc_all(p, bytes, 4)) return false;
    }
    const int nb = nblocks(L.nc);
    uint32_t *pk = nt ? (uint32_t *)p[0] : nullptr;
    int32_t *key = nt ? nullptr : (int32_t *)p[0], *pm = (int32_t *)(nt ? p[2] : p[3]);
    double *sS = nt ? nullptr : (double *)p[1], *sw = nt ? nullptr : (double *)p[2];
    if (D == 2)
        hipLaunchKernelGGL(build_slots64<2>, dim3(nb), dim3(kBlock), 0, stream, k64, (const uint16_t *)rec, 2 * nt, pk,
                           key, sS, sw, pm);
    else
        hipLaunchKernelGGL(build_slots64<3>, dim3(nb), dim3(kBlock), 0, stream, k64, (const uint16_t *)rec, 2 * nt, pk,
                           key, sS, sw, pm);
    if (rec) {
        (void)hipStreamSynchronize(stream);
        (void)hipFree(rec);
    }
    table64 = FaceTable<double>();
    k64.pk = pk;
    k64.pk_tab = nt ? (const double *)p[1] : nullptr;
    k64.sl_nb = key;
    k64.sl_S = sS;
    k64.sl_w = sw;
    k64.s_perm = pm;
    return true;
}

// the second state buffer of the one-launch stages (and the slots they
// read), allocated on first use; without them the step runs the separate
// launches, which compute the same bits
bool Solver::ensure_alt64() {
    if (!fused_ok) return false;
    if (q_alt64) return true;
    void *p = nullptr;
    const size_t bytes = (size_t)(L.D + 2) * ((size_t)L.nc + L.ng) * sizeof(double);
    fused_ok = ensure_slots64();
    if (fused_ok) fused_ok = alloc_all(&p, &bytes, 1);
    q_alt64 = (double *)p;
    return fused_ok;
}

bool Solver::ensure_alt32() {
    if (!fused_ok) return false;
    if (q_alt32) return true;
    if (!ensure_slots32()) {
        fused_ok = false;
        return false;
    }
    const size_t nq = (size_t)(L.D + 2) * ((size_t)L.nc + L.ng);
    void *p = nullptr;
    if (hipMalloc(&p, nq * sizeof(float)) != hipSuccess) {
        (void)hipGetLastError();
        fused_ok = false;
        return false;
    }
    allocs.push_back(p);
    device_bytes += (int64_t)(nq * sizeof(float));
    q_alt32 = (float *)p;
    return true;
}

// the first stage run as one fused launch (nstages when none is): every
// stage, except a residual stage 0, which keeps the separate launches for
// its per-block sums
int Solver::fused_from() const {
    if (!fused_ok || post_forces) return nstages;
    const int first = prm.have_res ? 1 : 0;
    return first < nstages ? first : nstages;
}

void Solver::stage_fused(int rk, bool from_alt) {
    stage_a(rk);  // the ghost fill after an outside write (no gradients here)
    auto launch = [&](const CflJob *job, bool fin) {
        if (!fp32) {
            double *qin = from_alt ? q_alt64 : k64.q, *qout = from_alt ? k64.q : q_alt64;
            LFM_DISPATCH_D(this, launch_stage_fused64<2>(this, A[rk], B[rk], dq_mode(rk), qin, qout, job, fin),
                           launch_stage_fused64<3>(this, A[rk], B[rk], dq_mode(rk), qin, qout, job, fin));
            return;
        }
        float *qin = from_alt ? q_alt32 : k32->q, *qout = from_alt ? k32->q : q_alt32;
        LFM_DISPATCH_D(this, launch_stage_fused32<2>(this, A[rk], B[rk], dq_mode(rk), qin, qout, job, fin),
                       launch_stage_fused32<3>(this, A[rk], B[rk], dq_mode(rk), qin, qout, job, fin));
    };
    if (rk == nstages - 1) {
        const CflJob job = cfl_job(true);
        prof_mark(5, true);
        launch(&job, false);
        prof_mark(5, false);
        final_or_carry(job);
        cfl_fused = true;
    } else {
        // a carried reduction is taken by the step's first stage
        const bool fin = cfl_pending && carry_target() == 1;
        if (fin) cfl_pending = false;
        prof_mark(3, true);
        launch(nullptr, fin);
        prof_mark(3, false);
    }
}

// the launch of a step that can take the previous step's carried CFL
// reduction before anything writes the reduction scratch: 1, the first
// one-launch stage (not a residual stage, and not the only stage, which
// forms the CFL itself); 2, the first FP32 gradient launch (each stage of a
// viscous or M2AUSM solver has one, before its update); 0, none
int Solver::carry_target() const {
    if (!L.halo.empty()) return 0;
    if (fused_ok) return have_alt() && fused_from() == 0 && nstages > 1 ? 1 : 0;
    return fp32 && (visc || prm.solver == 2) ? 2 : 0;
}

// the final reduction of a CFL job the last stage formed: carried into the
// next step (compute_cfl inside a run that steps again) or launched now
void Solver::final_or_carry(const CflJob &job) {
    if (defer_cfl && job.mode == 1 && job.out == d_cfl && carry_target() != 0) {
        cfl_pending = true;
        return;
    }
    prof_mark(4, true);
    cfl_final(job);
    prof_mark(4, false);
}

void Solver::flush_cfl() {
    if (!cfl_pending) return;
    cfl_pending = false;
    prof_mark(4, true);
    cfl_final(CflJob{1, dt, d_cfl, nullptr});
    prof_mark(4, false);
}

// one full time step (Mesh::solve loop body), no host synchronisation
void Solver::step() {
    const int first = fused_ok && ensure_alt() ? fused_from() : nstages;
    if (carry_target() == 0) flush_cfl();
    for (int rk = 0; rk < first; rk++) {
        stage_a(rk);
        stage_b(rk, true, true);
    }
    bool in_alt = false;
    for (int rk = first; rk < nstages; rk++) {
        stage_fused(rk, in_alt);
        in_alt = !in_alt;
    }
    // an odd number of one-launch stages left the state in the second
    // buffer: it becomes the state buffer (kernels take k32 by value at
    // launch, so later launches see the swap)
    if (in_alt) fp32 ? std::swap(k32->q, q_alt32) : std::swap(k64.q, q_alt64);
    end_step(true);
    eager_launches += nstages * (first < nstages ? 1 : 3) + 1;
}

// ---------------------------------------------------------------------------
// Steps as a graph.  A launch costs 2.7 us of host time and 3.6 us
// from one small kernel to the next; inside a graph of 40 kernels or more the
// next one starts after 1.8 (4 blocks) to 2.4 us (256 blocks).  A graph of one
// step's five launches gains nothing (3.7 us per kernel), so it holds
// kGraphSteps steps.  Building it costs what it saves in some 500 launches: it is
// done by a run that continues past kGraphAfter of them, and, where it could not
// be had, tried again after twice as many.
// ---------------------------------------------------------------------------
constexpr long kGraphAfter = 512;

struct Solver::StepGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    // all that its launches depend on
    KArgs k64;
    KArgs32 k32;
    const void *alt = nullptr;
    double dt = 0.0;
    bool pending = false;
    int from = 0;
    void note(const Solver &s) {
        std::memcpy((void *)&k64, &s.k64, sizeof k64);
        if (s.k32) std::memcpy((void *)&k32, s.k32, sizeof k32);
        alt = s.fp32 ? (const void *)s.q_alt32 : (const void *)s.q_alt64;
        dt = s.dt;
        pending = s.cfl_pending;
        from = s.fused_from();
    }
    bool matches(const Solver &s) const {
        return std::memcmp(&k64, &s.k64, sizeof k64) == 0 && (!s.k32 || std::memcmp(&k32, s.k32, sizeof k32) == 0) &&
               alt == (s.fp32 ? (const void *)s.q_alt32 : (const void *)s.q_alt64) && dt == s.dt &&
               pending == s.cfl_pending && from == s.fused_from();
    }
    ~StepGraph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};

void Solver::free_step_graph() {
    delete step_graph;
    step_graph = nullptr;
}

// whether the next kGraphSteps steps are one graph launch
bool Solver::graph_ready() {
    if (post || prof || ghosts_stale || nstages == 0) return false;
    // a step leaves its CFL reduction to the next one wherever it can: the
    // steps before the first such step are launched one by one
    if (!prm.adjust_dt && carry_target() != 0 && !cfl_pending) return false;
    if (step_graph && step_graph->matches(*this)) {
        graph_misses = 0;
        return true;
    }
    // an odd number of one-launch stages swaps the buffers each step: the
    // graph's turn comes with the next one
    if (step_graph && ++graph_misses < 2) return false;
    return eager_launches >= std::max(kGraphAfter, graph_after) && graph_build();
}

bool Solver::graph_build() {
    if (step_graph) {
        // its replays may still be queued: they read what it holds
        if (hipStreamSynchronize(stream) != hipSuccess) return false;
        free_step_graph();
    }
    auto g = std::make_unique<StepGraph>();
    g->note(*this);
    GraphBuild build;
    building = &build;
    const int64_t done = steps_done;
    defer_cfl = drop_dq = true;
    for (int i = 0; i < kGraphSteps; i++) step();
    steps_done = done;
    building = nullptr;
    eager_launches = 0;
    graph_misses = 0;
    if (build.finish(&g->graph, &g->exec) != hipSuccess || !g->matches(*this)) {
        // nothing was launched: the steps follow as launches of their own
        graph_after = 2 * std::max(kGraphAfter, graph_after);
        return false;
    }
    graph_after = 0;
    step_graph = g.release();
    return true;
}

int Solver::run_steps(int n, bool with_post) {
    if (n > 0)
        if (int rc = ensure_step_keys()) return rc;
    for (int i = 0; i < n;) {
        // the run's last step is never in the graph: it reduces its own CFL
        if (n - i > kGraphSteps && graph_ready()) {
            HIP_TRY(hipGraphLaunch(step_graph->exec, stream));
            steps_done += kGraphSteps;
            replayed_steps += kGraphSteps;
            if (prm.have_res) res_valid = true;
            i += kGraphSteps;
            continue;
        }
        defer_cfl = i + 1 < n && !(with_post && post);
        drop_dq = i + 1 < n;
        step();
        if (with_post && post) {
            const int rc = post_step();
            if (rc) {
                drop_dq = false;
                return rc;
            }
        }
        i++;
    }
    flush_cfl();
    return LFM_OK;
}

}  // namespace lfm

using lfm::fail;
using lfm::Solver;


extern "C" {

const char *lfm_last_error(void) { return lfm::g_last_error.c_str(); }

int lfm_solver_create(const lfm_polymesh *mesh, const lfm_params *prm, const double *p, const double *T,
                      const double *U3, const double *alpha, lfm_solver **out) {
    return lfm_solver_create_part(mesh, nullptr, prm, p, T, U3, alpha, out);
}

int lfm_solver_create_part(const lfm_polymesh *mesh, const lfm_partition *part, const lfm_params *prm,
                           const double *p, const double *T, const double *U3, const double *alpha,
                           lfm_solver **out) {
    if (!mesh || !prm || !p || !T || !U3 || !out) return fail(LFM_EINVAL, "null argument");
    *out = nullptr;
    if (prm->solver < 0 || prm->solver > 2) return fail(LFM_EINVAL, "solver must be 0 (M1), 1 (M2) or 2 (M2AUSM)");
    if (prm->rk_order < 0 || prm->rk_order > 5) return fail(LFM_EINVAL, "rkOrder must be 0..5");
    if (prm->precision != LFM_PREC_FP64 && prm->precision != LFM_PREC_FP32P)
        return fail(LFM_EINVAL, "precision must be 64 or 32");
    auto s = std::make_unique<Solver>();
    s->prm = *prm;
    std::string err;
    try {
        err = lfm::build_layout(*mesh, part, *prm, p, T, U3, alpha, s->L);
    } catch (const std::bad_alloc &) {
        return fail(LFM_ENOMEM, "out of host memory building the solver layout");
    } catch (const std::exception &e) {
        return fail(LFM_EINVAL, std::string("building the solver layout: ") + e.what());
    }
    if (!err.empty()) return fail(LFM_EINVAL, err);
    s->gas = lfm::derive_gas(*prm);
    s->nstages = lfm::rk_tables(prm->rk_order, s->A, s->B);
    s->dt = prm->dt;
    s->fp32 = prm->precision == LFM_PREC_FP32P;
    // the Smagorinsky stress does not scale with mu
    s->visc = prm->mu != 0.0 || !prm->laminar;
    HIP_TRY(hipGetDevice(&s->device));
    HIP_TRY(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
    HIP_TRY(hipEventCreate(&s->ev0));
    HIP_TRY(hipEventCreate(&s->ev1));
    HIP_TRY(hipHostMalloc((void **)&s->h_scalar, Solver::kScalars * sizeof(double) + Solver::kSmallRead,
                          hipHostMallocDefault));
    int rc = s->fp32 ? lfm::create_fp32p(s.get()) : lfm::create_fp64(s.get());
    if (rc) return rc;
    if (lfm::dev_upload(s.get(), (int32_t **)&s->d_comb, s->L.comb.data(), s->L.comb.size())) return LFM_EDEVICE;
    s->size_stage();
    s->halo_dev.resize(s->L.halo.size());
    for (size_t i = 0; i < s->L.halo.size(); i++) {
        const auto &hn = s->L.halo[i];
        auto &hd = s->halo_dev[i];
        hd.n_send = (int)hn.send_cells.size();
        hd.n_recv = (int)hn.ghost.size();
        std::vector<int32_t> gslot(hn.ghost.size());
        for (size_t j = 0; j < hn.ghost.size(); j++) gslot[j] = s->L.nc + hn.ghost[j];
        if (lfm::dev_upload(s.get(), &hd.send_cells, hn.send_cells.data(), hn.send_cells.size()) ||
            lfm::dev_upload(s.get(), &hd.recv_ghost, gslot.data(), gslot.size()) ||
            lfm::dev_zeros(s.get(), &hd.recv_src, gslot.size()))
            return LFM_EDEVICE;
    }
    if (s->slab_flush()) return LFM_EDEVICE;
    s->slab_host.reset();
    s->slab = nullptr;  // what follows is allocated by itself
    HIP_TRY(hipDeviceSynchronize());
    auto *h = new lfm_solver;
    h->impl = std::move(s);
    *out = h;
    return LFM_OK;
}

int lfm_solver_destroy(lfm_solver *h) {
    if (!h) return LFM_OK;
    if (h->impl && h->impl->stream) (void)hipStreamSynchronize(h->impl->stream);
    delete h;
    return LFM_OK;
}

int lfm_get_info(lfm_solver *h, lfm_info *info) {
    if (!h || !info) return fail(LFM_EINVAL, "null argument");
    Solver *s = h->impl.get();
    // one wait for the stream's work and the scalars behind it
    hipLaunchKernelGGL(lfm::export_scalars, dim3(1), dim3(64), 0, s->stream, s->d_scalar, 16, s->h_scalar);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    info->dim = s->L.D;
    info->n_cells = s->L.nc;
    info->n_cells_sm0 = s->L.nsm0;
    info->n_faces = s->L.nf;
    info->n_ghosts = s->L.ng;
    info->max_faces_per_cell = s->L.max_faces;
    info->precision = s->prm.precision;
    info->solver = s->prm.solver;
    info->device_bytes = s->device_bytes;
    info->dt = s->h_scalar[0];
    info->cfl = s->h_scalar[8];
    info->steps_done = s->steps_done;
    return LFM_OK;
}

int lfm_prepare_for_timestep(lfm_solver *h) {
    if (!h) return fail(LFM_EINVAL, "null handle");
    Solver *s = h->impl.get();
    s->zero_state_for_step();
    HIP_TRY(hipGetLastError());
    return LFM_OK;
}

int lfm_prepare_for_rkstep(lfm_solver *h, int rk) {
    if (!h) return fail(LFM_EINVAL, "null handle");
    Solver *s = h->impl.get();
    if (rk < 0 || rk >= std::max(1, s->nstages) || rk > 4) return fail(LFM_EINVAL, "rk stage out of range");
    s->pending_A = s->A[rk];
    s->pending_rk = rk;
    return LFM_OK;
}

int lfm_set_boundary_conditions(lfm_solver *h) {
    if (!h) return fail(LFM_EINVAL, "null handle");
    // the update kernel leaves the boundary ghosts as this fill would: it is
    // launched after the state was set from outside
    if (h->impl->ghosts_stale) h->impl->bc();
    h->impl->ghosts_stale = false;
    if (h->impl->post_forces) h->impl->post_snapshot();
    HIP_TRY(hipGetLastError());
    return LFM_OK;
}

int lfm_calc_gradients(lfm_solver *h) {
    // Gradients are produced together with the viscous terms by the same
    // cell gather (lfm_calc_vis); calling this alone is a no-op.
    if (!h) return fail(LFM_EINVAL, "null handle");
    return LFM_OK;
}

int lfm_calc_vis(lfm_solver *h) {
    if (!h) return fail(LFM_EINVAL, "null handle");
    if (!h->impl->halo_ready()) return fail(LFM_ESTATE, "halo set-up not imported for every neighbour");
    if (int rc = h->impl->ensure_keys(true)) return rc;
    h->impl->gradvis(true);
    HIP_TRY(hipGetLastError());
    return LFM_OK;
}

int lfm_one_rk_step(lfm_solver *h, int rk, double dt, double *res) {
    if (!h) return fail(LFM_EINVAL, "null handle");
    Solver *s = h->impl.get();
    if (rk < 0 || rk > 4) return fail(LFM_EINVAL, "rk stage out of range");
    if (!s->halo_ready()) return fail(LFM_ESTATE, "halo set-up not imported for every neighbour");
    if (int rc = s->ensure_keys(false)) return rc;
    const double B = s->B[rk];
    // without adjustTimeStep nothing on the device writes its deltaT, which
    // is then the last one that was set there.  The value goes with the
    // launch: a copy from host scratch may run after a later call's value is
    // in it.
    if (s->prm.adjust_dt || !(dt == s->dt)) {
        hipLaunchKernelGGL(lfm::set_scalar, dim3(1), dim3(64), 0, s->stream, s->d_dt_ptr(), dt);
        s->dt = dt;
    }
    const bool want_res = res && rk == 0 && s->prm.have_res;
    s->flux();
    s->update(s->pending_A, B, 0, want_res, false);
    s->pending_A = 1.0;
    HIP_TRY(hipGetLastError());
    if (want_res) {
        HIP_TRY(hipMemcpyAsync(s->h_scalar + 16, s->d_res, (s->L.D + 2) * sizeof(double), hipMemcpyDeviceToHost,
                               s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
        for (int k = 0; k < s->L.D + 2; k++) res[k] += s->h_scalar[16 + k];
        s->res_valid = true;
    }
    return LFM_OK;
}

int lfm_compute_dt(lfm_solver *h, double max_co, double *dt_out) {
    if (!h || !dt_out) return fail(LFM_EINVAL, "null argument");
    Solver *s = h->impl.get();
    if (s->fp32)  // FP64 sums over the slot lists
        if (int rc = s->ensure_keys(false)) return rc;
    s->cfl_dt(0, max_co, s->d_dtmin, s->h_scalar + 9);  // pinned: the kernel writes it there as well
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    *dt_out = s->h_scalar[9];
    return LFM_OK;
}

int lfm_compute_cfl(lfm_solver *h, double dt, double *cfl_out) {
    if (!h || !cfl_out) return fail(LFM_EINVAL, "null argument");
    Solver *s = h->impl.get();
    if (s->fp32)  // FP64 sums over the slot lists
        if (int rc = s->ensure_keys(false)) return rc;
    s->cfl_dt(1, dt, s->d_cfl, s->h_scalar + 8);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    *cfl_out = s->h_scalar[8];
    return LFM_OK;
}

int lfm_run(lfm_solver *h, int nsteps) {
    if (!h || nsteps < 0) return fail(LFM_EINVAL, "bad argument");
    Solver *s = h->impl.get();
    if (!s->L.halo.empty())
        return fail(LFM_ESTATE, "a partition with processor patches steps through lfm_part_group_run or the "
                                "per-stage calls with halo exchange");
    const int rc = s->run_steps(nsteps, true);
    if (rc) return rc;
    HIP_TRY(hipGetLastError());
    return LFM_OK;
}

int lfm_replayed_steps(lfm_solver *h, int64_t *n) {
    if (!h || !n) return fail(LFM_EINVAL, "null argument");
    *n = h->impl->replayed_steps;
    return LFM_OK;
}

int lfm_synchronize(lfm_solver *h) {
    if (!h) return fail(LFM_EINVAL, "null handle");
    HIP_TRY(hipStreamSynchronize(h->impl->stream));
    return LFM_OK;
}

int lfm_time_steps(lfm_solver *h, int nsteps, double *ms_out) {
    if (!h || !ms_out || nsteps < 0) return fail(LFM_EINVAL, "bad argument");
    Solver *s = h->impl.get();
    if (!s->L.halo.empty())
        return fail(LFM_ESTATE, "a partition with processor patches steps through lfm_part_group_run or the "
                                "per-stage calls with halo exchange");
    HIP_TRY(hipEventRecord(s->ev0, s->stream));
    const int rc = s->run_steps(nsteps, false);
    if (rc) return rc;
    HIP_TRY(hipEventRecord(s->ev1, s->stream));
    HIP_TRY(hipEventSynchronize(s->ev1));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, s->ev0, s->ev1));
    *ms_out = ms;
    return LFM_OK;
}

int lfm_profile_steps(lfm_solver *h, int nsteps, double *ms_per_group, double *ms_total) {
    if (!h || !ms_per_group || !ms_total || nsteps < 1) return fail(LFM_EINVAL, "bad argument");
    Solver *s = h->impl.get();
    if (!s->L.halo.empty())
        return fail(LFM_ESTATE, "a partition with processor patches steps through lfm_part_group_run or the "
                                "per-stage calls with halo exchange");
    if (int rc = s->ensure_step_keys()) return rc;
    const size_t need = (size_t)nsteps * (s->nstages * 8 + 2);
    for (hipEvent_t e : s->prof_ev) (void)hipEventDestroy(e);
    s->prof_ev.assign(need, nullptr);
    s->prof_grp.assign(need, 0);
    for (size_t i = 0; i < need; i++) HIP_TRY(hipEventCreate(&s->prof_ev[i]));
    s->prof_n = 0;
    s->prof = true;
    HIP_TRY(hipEventRecord(s->ev0, s->stream));
    for (int i = 0; i < nsteps; i++) {
        s->defer_cfl = i + 1 < nsteps;
        s->step();
    }
    s->flush_cfl();
    HIP_TRY(hipEventRecord(s->ev1, s->stream));
    s->prof = false;
    HIP_TRY(hipEventSynchronize(s->ev1));
    for (int g = 0; g < Solver::kProfGroups; g++) ms_per_group[g] = 0.0;
    for (size_t i = 0; i + 1 < s->prof_n; i += 2) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, s->prof_ev[i], s->prof_ev[i + 1]));
        const int g = s->prof_grp[i];
        if (g >= 0 && g < Solver::kProfGroups) ms_per_group[g] += ms;
    }
    float tot = 0.f;
    HIP_TRY(hipEventElapsedTime(&tot, s->ev0, s->ev1));
    *ms_total = tot;
    for (hipEvent_t e : s->prof_ev) (void)hipEventDestroy(e);
    s->prof_ev.clear();
    s->prof_grp.clear();
    return LFM_OK;
}

int lfm_get_field(lfm_solver *h, int which, double *out) {
    if (!h || !out) return fail(LFM_EINVAL, "null argument");
    return h->impl->get_field(which, out);
}

int lfm_set_field(lfm_solver *h, int which, const double *in) {
    if (!h || !in) return fail(LFM_EINVAL, "null argument");
    return h->impl->set_field(which, in);
}

int lfm_get_residual(lfm_solver *h, double *res) {
    if (!h || !res) return fail(LFM_EINVAL, "null argument");
    Solver *s = h->impl.get();
    HIP_TRY(hipMemcpyAsync(s->h_scalar + 16, s->d_res, (s->L.D + 2) * sizeof(double), hipMemcpyDeviceToHost,
                           s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    for (int k = 0; k < s->L.D + 2; k++) res[k] = s->h_scalar[16 + k];
    return LFM_OK;
}

int lfm_conservation(lfm_solver *h, double *out) {
    if (!h || !out) return fail(LFM_EINVAL, "null argument");
    Solver *s = h->impl.get();
    lfm::integrals(s, s->d_scalar + 10);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(s->h_scalar + 24, s->d_scalar + 10, (s->L.D + 2) * sizeof(double), hipMemcpyDeviceToHost,
                           s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    for (int k = 0; k < s->L.D + 2; k++) out[k] = s->h_scalar[24 + k];
    return LFM_OK;
}

int lfm_check_finite(lfm_solver *h, int64_t *n_bad) {
    if (!h || !n_bad) return fail(LFM_EINVAL, "null argument");
    return h->impl->check_finite(n_bad);
}

int lfm_check_finite_noalloc(lfm_solver *h, int64_t *n_bad) {
    if (!h || !n_bad) return fail(LFM_EINVAL, "null argument");
    return h->impl->check_finite_noalloc(n_bad);
}

}  // extern "C"
